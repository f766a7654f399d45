"""The workloads this engine is measured on: prompts and decode steps through ``ModelRunner.step``.

Every case is one model with seeded random weights behind the engine's step function, as a serving program
drives it: ``random_model`` makes the model, ``ModelRunner`` owns its cache, ``step`` runs batches of
(request, its next tokens) and returns logits.  Three kinds of pass:

* ``prompt``: requests begin, their whole prompts run as ONE step, the logits of each last token come back,
  the requests end (time to first token of one prompt, or of several that arrive together);
* ``decode``: one step of one token per request behind the tokens each holds in the cache (the contexts grow by
  one token a pass, as they do in use; a batch that reaches its length begins anew);
* ``serve``: a prompt arrives while others decode: it runs in portions, every step a portion beside one token of
  every decoding request.

Widths, heads, ranks, experts and vocabularies are those of ``bench.py`` (Mistral 7B with and without a window, 12B,
24B; Bugidra and Fipitar at two widths); the Mistral cases run the first few of the model's equal layers, so that a
state is made quickly.  Caches are filled by running prompts.  Bugidra and Fipitar stand for the designs with
recurrences, latent attention and side-by-side mixers; designs with routed experts are left out, because a router's
near-tie that rounding decides changes an expert, and two correct runs in bfloat16 then differ by several percent.  ``exact`` computes the same logits in 64 bits with
plain torch, the weights drawn by the rule that ``flambeau_amd/weights/random_init.py`` states.
"""
from __future__ import annotations

import hashlib
import math
import random

import torch

_MISTRAL = {"architectures": ["MistralForCausalLM"], "model_type": "mistral", "hidden_act": "silu", "rms_norm_eps": 1e-5,
            "max_position_embeddings": 32768, "tie_word_embeddings": False, "num_attention_heads": 32, "num_key_value_heads": 8,
            "head_dim": 128}
MISTRAL_SIZES = {
    "7b": dict(_MISTRAL, hidden_size=4096, intermediate_size=14336, vocab_size=32768, rope_theta=1e6, sliding_window=None),
    "v01": dict(_MISTRAL, hidden_size=4096, intermediate_size=14336, vocab_size=32000, rope_theta=1e4, sliding_window=4096),
    "12b": dict(_MISTRAL, hidden_size=5120, intermediate_size=14336, vocab_size=131072, rope_theta=1e6, sliding_window=None),
    "24b": dict(_MISTRAL, hidden_size=5120, intermediate_size=32768, vocab_size=131072, rope_theta=1e8, sliding_window=None),
}
BUGIDRA_SIZES = {
    "w2048": dict(width=2048, heads=16, kv_heads=8, ff=8192, ret_heads=8, delta_heads=16, delta_qk_heads=8),
    "w4096": dict(width=4096, heads=32, kv_heads=8, ff=14336, ret_heads=16, delta_heads=32, delta_qk_heads=16),
}
FIPITAR_SIZES = {
    "w2048": dict(width=2048, heads=16, kv_heads=8, ff=8192, ret_heads=8, gla_heads=16, q_rank=768, kv_rank=256),
    "w4096": dict(width=4096, heads=32, kv_heads=8, ff=14336, ret_heads=16, gla_heads=32, q_rank=1536, kv_rank=512),
}
VOCAB = 32768              # of the two designs
PAGE = 16
LAYERS_DESIGN = 6


def _bugidra(s):
    att = {"type": "attention", "mixer": dict(heads=s["heads"], kv_heads=s["kv_heads"], dim=128, vdim=128, scale=128 ** -0.5, softcap=50.0,
                                              v_mix=True, rot={"base": 10000.0, "dims": 64})}
    left = dict(heads=s["heads"], kv_heads=s["kv_heads"], dim=128, vdim=128, scale=0.09,
                rot={"base": 50000.0, "dims": 128, "scaling": {"factor": 2.0, "original": 4096, "fast": 32.0, "slow": 1.0}})
    right = dict(heads=s["ret_heads"], dim=128, vdim=128, decay=[1.0 - 2.0 ** -(5 + i % 8) for i in range(s["ret_heads"])],
                 rot={"base": 1e6, "dims": 128})
    par = {"type": "parallel", "mixer": {"left": left, "right": right}}
    delta = {"type": "delta", "mixer": dict(heads=s["delta_heads"], kv_heads=s["delta_qk_heads"], dim=128, vdim=128, conv=4)}
    mlp = {"kind": "dense", "ff": s["ff"]}
    return {"architecture": "Bugidra", "vocab": VOCAB, "width": s["width"], "norm": {"eps": 1e-5}, "embedding": {"scale": s["width"] ** 0.5},
            "layers": [dict(layer, mlp=mlp) for layer in (delta, par, att, delta, par, att)]}


def _fipitar(s):
    gla = {"type": "gla", "mixer": dict(heads=s["gla_heads"], dim=128, vdim=128, tau=16.0, decay_rank=64)}
    latent = {"type": "latent_attention", "mixer": dict(
        heads=s["heads"], dim=128, rot_dim=64, vdim=128, q_rank=s["q_rank"], kv_rank=s["kv_rank"], scale=192 ** -0.5,
        rot={"base": 1e6, "dims": 64, "scaling": {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}})}
    left = dict(heads=s["heads"], kv_heads=s["kv_heads"], dim=128, vdim=128, scale=128 ** -0.5, softcap=50.0, rot={"base": 50000.0, "dims": 64})
    right = dict(heads=2 * s["ret_heads"], vdim=64, state=128, groups=8, conv=4, norm_groups=8)
    par = {"type": "parallel", "mixer": dict(left=left, right=right, left_scale=0.8, right_scale=1.2)}
    mlp = {"kind": "dense", "ff": s["ff"], "limit": 7.0}
    return {"architecture": "Fipitar", "vocab": VOCAB, "width": s["width"], "norm": {"eps": 1e-5},
            "layers": [dict(layer, mlp=mlp) for layer in (gla, par, latent, gla, par, latent)]}


def config_of(case):
    if case["design"] == "fipitar":
        return _fipitar(FIPITAR_SIZES[case["size"]])
    if case["design"] == "bugidra":
        return _bugidra(BUGIDRA_SIZES[case["size"]])
    return dict(MISTRAL_SIZES[case["size"]], num_hidden_layers=case["layers"])


def vocab_of(case):
    return MISTRAL_SIZES[case["size"]]["vocab_size"] if case["design"] == "mistral" else VOCAB


# ---------------------------------------------------------------- the cases
def _case(name, design, size, kind, layers, batch, shortest, longest, dtype="bfloat16", portion=0, portions=0):
    """``batch`` requests whose prompts (or cached contexts) are ``shortest`` to ``longest`` tokens long; ``serve`` has
    ``portions`` portions of ``portion`` tokens beside them."""
    c = dict(design=design, size=size, kind=kind, layers=layers, dtype=dtype, batch=batch, shortest=shortest, longest=longest,
             portion=portion, portions=portions)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one user's chat: every token waits for this step; launches and the weights' first bytes count
        _case("decode_1", "mistral", "7b", "decode", 8, 1, 2048, 2048),
        # a small server, the workload that bench.py reports first; contexts of unlike lengths
        _case("decode_8", "mistral", "7b", "decode", 8, 8, 1000, 4100),
        # a full server: the largest batch of the serving workloads, contexts from a question to a long document
        _case("decode_64", "mistral", "7b", "decode", 4, 64, 128, 4096),
        # a few short questions that arrive together: too many rows for the decode kernels, too few to fill the chip
        _case("prompts_short", "mistral", "7b", "prompt", 4, 3, 45, 131),
        # time to first token of a document, the prefill that bench.py reports
        _case("prompt_2048", "mistral", "7b", "prompt", 4, 1, 2048, 2048),
        # the largest dense model of the configurations with a long prompt
        _case("prompt_24b", "mistral", "24b", "prompt", 4, 1, 4001, 4001),
        # a prompt of 2,048 tokens in portions of 512 while 16 others decode, window of 4,096 (what the scheduler builds)
        _case("serve_window", "mistral", "v01", "serve", 4, 16, 500, 6000, portion=512, portions=4),
        # the 32-bit path, what a trace is checked with: a prompt of some hundred tokens, then token by token
        _case("float32_prompt", "mistral", "7b", "prompt", 2, 1, 333, 333, dtype="float32"),
        _case("float32_decode", "mistral", "7b", "decode", 2, 1, 340, 340, dtype="float32"),
        # the design with the delta rule, retention and gated attention: a prompt, and a small server
        _case("bugidra_prompt", "bugidra", "w4096", "prompt", LAYERS_DESIGN, 1, 2048, 2048),
        _case("bugidra_decode", "bugidra", "w4096", "decode", LAYERS_DESIGN, 8, 500, 2500),
        # the design with gated linear attention, a state space and latent attention: a prompt
        _case("fipitar_prompt", "fipitar", "w4096", "prompt", LAYERS_DESIGN, 1, 2048, 2048),
    ]


def _spread(rng, lo, hi):
    """A whole number between ``lo`` and ``hi``, spread evenly over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "serve", "design", "design", "float32"])
    if kind == "design":
        design, size, layers = rng.choice(["bugidra", "fipitar"]), rng.choice(["w2048", "w4096"]), LAYERS_DESIGN
        if rng.random() < 0.5:
            n = _spread(rng, 30, 2048)
            return _case(None, design, size, "prompt", layers, 1, n, n)
        longest = _spread(rng, 300, 3000)
        return _case(None, design, size, "decode", layers, _spread(rng, 1, 16), _spread(rng, 60, longest), longest)
    if kind == "float32":
        if rng.random() < 0.5:
            n = _spread(rng, 9, 333)
            return _case(None, "mistral", rng.choice(["7b", "v01"]), "prompt", 2, 1, n, n, dtype="float32")
        n = _spread(rng, 30, 600)
        return _case(None, "mistral", "7b", "decode", 2, rng.randint(1, 4), n, n, dtype="float32")
    size = rng.choice(["7b", "7b", "v01", "12b", "24b"])
    if kind == "decode":
        batch = _spread(rng, 1, 64)
        longest = _spread(rng, 300, 4096 if batch > 8 else 12000)
        return _case(None, "mistral", size, "decode", 4, batch, _spread(rng, 100, longest), longest)
    if kind == "prompt":
        batch = rng.choice([1, 1, 1, 2, 4])
        longest = _spread(rng, 17, 4000 // batch)
        return _case(None, "mistral", size, "prompt", rng.randint(2, 4), batch, _spread(rng, 9, longest), longest)
    longest = _spread(rng, 300, 8000)
    return _case(None, "mistral", size, "serve", 2 if size == "24b" else 3, _spread(rng, 2, 32), _spread(rng, 100, longest), longest,
                 portion=rng.choice([128, 256, 512, 1024]), portions=rng.randint(1, 3))


def lengths_of(case):
    """Tokens of each request's prompt, or in its cache: fixed by the case, so that the work is."""
    rng = random.Random(f"{case['batch']} {case['shortest']} {case['longest']}")
    return [_spread(rng, case["shortest"], case["longest"]) for _ in range(case["batch"])]


def passes_of(case):
    """Passes that a state's contexts have room for before the requests begin anew."""
    return 4096 if case["kind"] == "decode" and case["batch"] <= 8 else 1024


def tokens_of(case, seed):
    """(the requests' prompts, the tokens they decode pass by pass, the prompt that arrives in portions)"""
    g = torch.Generator().manual_seed(int(seed) * 7919 + 17)
    ids = lambda n: torch.randint(0, vocab_of(case), (n,), generator=g).tolist()
    prompts = [ids(n) for n in lengths_of(case)]
    steps = max(case["portions"], 1)
    decoded = [ids(case["batch"]) for _ in range(passes_of(case) * steps if case["kind"] != "prompt" else 0)]
    return prompts, decoded, ids(case["portion"] * case["portions"])


# ---------------------------------------------------------------- a pass
class State:
    """What a serving program holds: the model, the runner with its cache, the requests' tokens."""


def prepare(case, seed):
    from flambeau_amd import ModelRunner, random_model
    s = State()
    s.case = case
    s.prompts, s.decoded, s.arriving = tokens_of(case, seed)
    longest = max(len(p) for p in s.prompts)
    most = sum(len(p) for p in s.prompts) if case["kind"] == "prompt" else max(2048, case["portion"] + case["batch"])
    s.model, _ = random_model(config_of(case), seed=int(seed), dtype=case["dtype"], max_batch_tokens=most, std=0.02, gain_std=0.0)
    room = longest + 1 + (len(s.decoded) if case["kind"] != "prompt" else 0)
    pages = lambda n: -(-n // PAGE) + 1
    n_pages = sum(pages(len(p) + room - longest) for p in s.prompts) + pages(len(s.arriving))
    s.runner = ModelRunner(s.model, n_pages=n_pages, page_size=PAGE, max_slots=case["batch"] + 1, max_seq_len=max(room, len(s.arriving) + 1),
                           max_logit_rows=case["batch"] + 1)
    if case["kind"] != "prompt":
        _fill(s)
    return s


def _fill(s):
    """Begin the decoding requests and run their prompts, in steps of up to 2,048 tokens."""
    from flambeau_amd import StepEntry
    s.at = 0
    batch, room = [], 2048
    for i, prompt in enumerate(s.prompts):
        if i in s.runner.manager.live:
            s.runner.end(i)
    for i, prompt in enumerate(s.prompts):
        s.runner.begin(i)
        for at in range(0, len(prompt), 2048):
            piece = prompt[at:at + 2048]
            if len(piece) > room or any(e.request_id == i for e in batch):
                s.runner.step(batch)
                batch, room = [], 2048
            batch.append(StepEntry(i, piece, []))
            room -= len(piece)
    s.runner.step(batch)


def run(s):
    from flambeau_amd import StepEntry
    case, runner = s.case, s.runner
    if case["kind"] == "prompt":
        for i in range(len(s.prompts)):
            runner.begin(i)
        logits = runner.step([StepEntry(i, p, [len(p) - 1]) for i, p in enumerate(s.prompts)])
        for i in range(len(s.prompts)):
            runner.end(i)
        return logits
    if s.at + max(case["portions"], 1) > len(s.decoded):
        _fill(s)
    if case["kind"] == "decode":
        logits = runner.step([StepEntry(i, [t], [0]) for i, t in enumerate(s.decoded[s.at])])
        s.at += 1
        return logits
    out, n = [], case["portion"]
    runner.begin("arriving")
    for k in range(case["portions"]):
        entries = [StepEntry(i, [t], [0]) for i, t in enumerate(s.decoded[s.at])]
        entries.append(StepEntry("arriving", s.arriving[k * n:(k + 1) * n], [n - 1] if k == case["portions"] - 1 else []))
        out.append(runner.step(entries).clone())          # (the next step writes over the buffer; a program would sample from it here)
        s.at += 1
    runner.end("arriving")
    return out


# ---------------------------------------------------------------- what a pass cannot do without
def _weights_of(case):
    """Matrix values of the layers: what a step reads of them, and multiplications per token."""
    if case["design"] == "mistral":
        c = MISTRAL_SIZES[case["size"]]
        h, hd = c["hidden_size"], c["head_dim"]
        per = (c["num_attention_heads"] + 2 * c["num_key_value_heads"]) * hd * h + c["num_attention_heads"] * hd * h + 3 * c["intermediate_size"] * h
        return case["layers"] * per
    if case["design"] == "fipitar":
        s = FIPITAR_SIZES[case["size"]]
        w, hd, kd, gd, inner = s["width"], s["heads"] * 128, s["kv_heads"] * 128, s["gla_heads"] * 128, 2 * s["ret_heads"] * 64
        gla = w * (5 * gd + 64) + 64 * gd
        pair = w * (2 * hd + 2 * kd + s["heads"]) + w * (3 * inner + 2 * 8 * 128 + 2 * s["ret_heads"])
        latent = w * (s["q_rank"] + s["kv_rank"] + 64 + hd) + s["q_rank"] * s["heads"] * 192 + 2 * hd * s["kv_rank"]
        return 2 * (gla + pair + latent) + LAYERS_DESIGN * 3 * w * s["ff"]
    s = BUGIDRA_SIZES[case["size"]]
    w, hd, kd, rd, dd, dk = s["width"], s["heads"] * 128, s["kv_heads"] * 128, s["ret_heads"] * 128, s["delta_heads"] * 128, s["delta_qk_heads"] * 128
    attention = w * (3 * hd + 2 * kd)
    pair = w * (2 * hd + 2 * kd) + 5 * w * rd
    delta = w * (2 * dk + 3 * dd + 2 * s["delta_heads"])
    return 2 * (attention + pair + delta) + LAYERS_DESIGN * 3 * w * s["ff"]


def _attention_of(case):
    """(cached values per token over all layers, flops per query and key over all of them)"""
    if case["design"] == "mistral":
        return case["layers"] * 2 * 8 * 128, case["layers"] * 4 * 32 * 128
    if case["design"] == "fipitar":
        s = FIPITAR_SIZES[case["size"]]
        return 2 * 2 * s["kv_heads"] * 128 + 2 * (s["kv_rank"] + 64), 2 * s["heads"] * (4 * 128 + 2 * 320)
    s = BUGIDRA_SIZES[case["size"]]
    return 4 * 2 * s["kv_heads"] * 128, 4 * 4 * s["heads"] * 128


def _recurrent(case):
    """(state values per request over all layers, flops per token over all of them)"""
    if case["design"] == "fipitar":
        s = FIPITAR_SIZES[case["size"]]
        gla, ssd = s["gla_heads"] * 128 * 128, 2 * s["ret_heads"] * 128 * 64
        return 2 * (gla + ssd), 2 * 5 * (gla + ssd)
    if case["design"] == "bugidra":
        s = BUGIDRA_SIZES[case["size"]]
        delta, ret = s["delta_heads"] * 128 * 128, s["ret_heads"] * 128 * 128
        return 2 * (delta + ret), 2 * (7 * delta + 5 * ret)
    return 0, 0


def work(case):
    el = 4 if case["dtype"] == "float32" else 2
    window = MISTRAL_SIZES[case["size"]]["sliding_window"] or 0 if case["design"] == "mistral" else 0
    hidden = config_of(case).get("hidden_size") or config_of(case)["width"]
    head, lengths = vocab_of(case) * hidden, lengths_of(case)
    seen = lambda p: min(p + 1, window) if window else p + 1                       # keys that a query at position p sees
    span = lambda a, n: sum(seen(p) for p in range(a, a + n))
    if case["kind"] == "prompt":
        steps = [[(0, n, 1) for n in lengths]]                                      # (first position, tokens, wanted rows)
    elif case["kind"] == "decode":
        steps = [[(n, 1, 1) for n in lengths]]
    else:
        steps = [[(n + k, 1, 1) for n in lengths] + [(k * case["portion"], case["portion"], int(k == case["portions"] - 1))]
                 for k in range(case["portions"])]
    cached, per_key = _attention_of(case)
    weights = _weights_of(case)
    state, state_flops = _recurrent(case)
    nbytes = flops = 0.0
    for step in steps:
        rows, wanted = sum(n for _, n, _ in step), sum(w for _, _, w in step)
        nbytes += el * (weights + head) + 4 * wanted * vocab_of(case)
        flops += 2.0 * rows * weights + 2.0 * wanted * head
        for at, n, _ in step:
            old = min(at, max(window - 1, 0)) if window else at
            nbytes += cached * el * (old + n) + 4 * state * (2 if at else 1)
            flops += per_key * float(span(at, n)) + state_flops * n
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # bfloat16: the logits are 1.4 to 2.1 % (Mistral) and 0.8 % (the designs) off those in 64 bits, nearly all of it from
    # the rounding of stored activations, which another order of the sums redraws; 32 bits: 8e-7 off
    if case["dtype"] == "float32":
        return {"rel": 4e-6}
    return {"rel": 0.03, "max": 0.3}


# ---------------------------------------------------------------- the same in 64 bits
class _Weights:
    """The random model's tensors, each from a generator of its own seeded with (seed, name): what
    ``flambeau_amd/weights/random_init.py`` says of them, rounded to the model's type, in 64 bits."""

    def __init__(self, case, seed):
        self.seed, self.dtype = int(seed), getattr(torch, case["dtype"])

    def _generator(self, name):
        at = int.from_bytes(hashlib.sha256(f"{self.seed}:{name}".encode()).digest()[:8], "little") & ((1 << 63) - 1)
        return torch.Generator(device="cuda").manual_seed(at)

    def matrix(self, name, *shape):
        x = torch.randn(shape, generator=self._generator(name), device="cuda", dtype=torch.float32) * 0.02
        return x.to(self.dtype).double()

    def uniform(self, name, lo, hi, *shape):
        x = lo + (hi - lo) * torch.rand(shape, generator=self._generator(name), device="cuda")
        return x.to(self.dtype).double()

    def alpha(self, name):
        x = torch.full((), 0.5, device="cuda") * (1.0 + 0.1 * torch.randn((), generator=self._generator(name), device="cuda"))
        return x.to(self.dtype).double()


def _rms(x, eps=1e-5):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _by_rows(x, f, n=8192):
    return torch.cat([f(x[i:i + n]) for i in range(0, x.shape[0], n)])


def _angles(n, rot):
    dims, base = rot["dims"], float(rot["base"])
    f = torch.tensor([base ** (-2.0 * i / dims) for i in range(dims // 2)], dtype=torch.float64, device="cuda")
    magnitude, sc = 1.0, rot.get("scaling")
    if sc:
        turn = lambda t: dims * math.log(sc["original"] / (2.0 * math.pi * t)) / (2.0 * math.log(base))
        lo, hi = max(math.floor(turn(sc["fast"])), 0), min(math.ceil(turn(sc["slow"])), dims - 1)
        ramp = ((torch.arange(dims // 2, dtype=torch.float64, device="cuda") - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
        f, magnitude = f / sc["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(sc["factor"]) + 1.0
    a = torch.arange(n, dtype=torch.float64, device="cuda")[:, None] * f[None, :]
    return (a.cos() * magnitude)[:, None, :], (a.sin() * magnitude)[:, None, :]


def _rotate(x, rot, interleaved=False):
    """x [T, heads, dim]: the first ``dims`` values of every head, in halves or in neighbouring pairs."""
    c, s = _angles(x.shape[0], rot)
    d, y = rot["dims"], x.clone()
    one, two = (slice(0, d, 2), slice(1, d, 2)) if interleaved else (slice(0, d // 2), slice(d // 2, d))
    u, v = x[..., one], x[..., two]
    y[..., one], y[..., two] = u * c - v * s, v * c + u * s
    return y


def _layer_norm(x, bias):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + 1e-5) + bias


def _short_convolution(z, weight, bias=None):
    """z [T, channels], weight [channels, taps]: the last tap belongs to the token itself, zeros before the start."""
    taps = weight.shape[1]
    out = torch.zeros_like(z) if bias is None else bias.repeat(z.shape[0], 1)
    for j in range(min(taps, z.shape[0])):
        out[j:] += z[:z.shape[0] - j] * weight[:, taps - 1 - j]
    return torch.nn.functional.silu(out)


def _attend(q, k, v, scale, window=0, softcap=None, sink=None, block=512):
    """q [T, H, D], k and v [T, G, D]: causal softmax attention, query head h reads key head h // (H / G); ``sink``, a
    score per head, joins the denominator."""
    T, H, _ = q.shape
    G = k.shape[1]
    kt, vt = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()         # [G, D, T], [G, T, Dv]
    out = torch.empty(T, H, v.shape[2], dtype=q.dtype, device=q.device)
    for a in range(0, T, block):
        b = min(T, a + block)
        lo = max(0, a - window + 1) if window else 0
        qs = q[a:b].permute(1, 0, 2).reshape(G, (H // G) * (b - a), -1)
        s = torch.matmul(qs, kt[:, :, lo:b].contiguous()).view(G, H // G, b - a, b - lo) * scale
        if softcap is not None:
            s = softcap * torch.tanh(s / softcap)
        i, j = torch.arange(a, b, device=q.device)[:, None], torch.arange(lo, b, device=q.device)[None, :]
        s.masked_fill_((j > i) | ((j <= i - window) if window else (j < 0)), -math.inf)
        if sink is not None:
            s = torch.cat([s, sink.view(G, H // G, 1, 1).expand(-1, -1, b - a, 1)], -1)
        o = torch.matmul(torch.softmax(s, -1)[..., :b - lo].reshape(G, -1, b - lo), vt[:, lo:b].contiguous())
        out[a:b] = o.view(H, b - a, -1).permute(1, 0, 2)
    return out.reshape(T, -1)


def _exact_mistral(case, W, tokens, lengths, wanted):
    c = MISTRAL_SIZES[case["size"]]
    h, hd, H, G, ff = c["hidden_size"], 128, 32, 8, c["intermediate_size"]
    x = W.matrix("model.embed_tokens.weight", c["vocab_size"], h)[tokens]
    rot = {"base": c["rope_theta"], "dims": hd}
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        y = _rms(x)
        q, k, v = (_by_rows(y, lambda r, w=W.matrix(p + f"self_attn.{n}_proj.weight", m * hd, h): r @ w.T).view(-1, m, hd)
                   for n, m in (("q", H), ("k", G), ("v", G)))
        o, at = torch.empty(x.shape[0], H * hd, dtype=x.dtype, device=x.device), 0
        for n in lengths:
            o[at:at + n] = _attend(_rotate(q[at:at + n], rot), _rotate(k[at:at + n], rot), v[at:at + n], hd ** -0.5, c["sliding_window"] or 0)
            at += n
        w = W.matrix(p + "self_attn.o_proj.weight", h, H * hd)
        x += _by_rows(o, lambda r: r @ w.T)
        del q, k, v, o, y
        gate, up, down = (W.matrix(p + f"mlp.{n}_proj.weight", *s) for n, s in (("gate", (ff, h)), ("up", (ff, h)), ("down", (h, ff))))
        x += _by_rows(_rms(x), lambda r: (torch.nn.functional.silu(r @ gate.T) * (r @ up.T)) @ down.T)
    return _rms(x[wanted]) @ W.matrix("lm_head.weight", c["vocab_size"], h).T


def _retention(q, k, v, decay, block=512):
    T, H, _ = q.shape
    q, k, v = (t.permute(1, 0, 2).contiguous() for t in (q, k, v))
    logs, out, kt = torch.log(decay)[:, None, None], torch.empty(T, H, v.shape[2], dtype=v.dtype, device=v.device), k.transpose(1, 2).contiguous()
    for a in range(0, T, block):
        b = min(T, a + block)
        i, j = torch.arange(a, b, device=q.device)[:, None], torch.arange(b, device=q.device)[None, :]
        s = torch.matmul(q[:, a:b], kt[:, :, :b].contiguous()) * torch.exp(logs * (i - j)).masked_fill(j > i, 0.0)
        out[a:b] = torch.matmul(s, v[:, :b].contiguous()).permute(1, 0, 2)
    return out


def _delta(q, k, v, g, beta):
    """S <- g S; u = beta (v - S^T k); S <- S + k u^T; o = S^T q, token by token for all heads of one sequence."""
    T, H, D = q.shape
    S, out = torch.zeros(H, D, v.shape[2], dtype=v.dtype, device=v.device), torch.empty_like(v)
    for t in range(T):
        S *= g[t, :, None, None]
        u = beta[t, :, None] * (v[t] - torch.matmul(k[t, :, None, :], S)[:, 0])
        S += k[t, :, :, None] * u[:, None, :]
        out[t] = torch.matmul(q[t, :, None, :], S)[:, 0]
    return out


def _exact_bugidra(case, W, tokens, lengths, wanted):
    s, cfg = BUGIDRA_SIZES[case["size"]], config_of(case)
    w, silu, sig = s["width"], torch.nn.functional.silu, torch.sigmoid
    x = W.matrix("embed", VOCAB, w)[tokens] * cfg["embedding"]["scale"]
    dyt = lambda x, n: torch.tanh(W.alpha(n + ".alpha") * x) + W.matrix(n + ".b", w)
    split = lambda f, *ts: torch.cat([f(*t) for t in zip(*(t.split(lengths) for t in ts))])
    first_values = None

    for i, layer in enumerate(cfg["layers"]):
        p, m, kind = f"l{i}.mix.", layer["mixer"], layer["type"]
        y = dyt(x, f"l{i}.norm1")
        lin = lambda n, rows, z=None: (y if z is None else z) @ W.matrix(p + n, rows, (y if z is None else z).shape[1]).T
        if kind == "attention":
            H, G = m["heads"], m["kv_heads"]
            q, k, v = _rms(lin("q", H * 128)).view(-1, H, 128), _rms(lin("k", G * 128)).view(-1, G, 128), lin("v", G * 128).view(-1, G, 128)
            if first_values is None:
                first_values = v
            else:
                mix = W.uniform(p + "vmix", 0.0, 1.0)
                v = (1.0 - mix) * v + mix * first_values
            o = split(lambda q, k, v: _attend(_rotate(q, m["rot"], True), _rotate(k, m["rot"], True), v, m["scale"], softcap=m["softcap"]), q, k, v)
            x = x + lin("o", w, o * sig(lin("g", H * 128)))
        elif kind == "parallel":
            a, b = m["left"], m["right"]
            H, G, R = a["heads"], a["kv_heads"], b["heads"]
            q, k, v = (lin("left." + n, d * 128).view(-1, d, 128) for n, d in (("q", H), ("k", G), ("v", G)))
            o = split(lambda q, k, v: _attend(_rms(_rotate(q, a["rot"])), _rms(_rotate(k, a["rot"])), v, a["scale"]), q, k, v)
            left = _rms(lin("left.o", w, o))
            q, k, v = (lin("right." + n, R * 128).view(-1, R, 128) for n in ("q", "k", "v"))
            decay = torch.tensor(b["decay"], dtype=torch.float64, device="cuda")
            o = split(lambda q, k, v: _retention(_rotate(q, b["rot"]), _rotate(k, b["rot"]) * 128 ** -0.5, v, decay), q, k, v)
            right = _rms(lin("right.o", w, _rms(o).reshape(-1, R * 128) * silu(lin("right.g", R * 128))))
            x = x + 0.5 * (left + right)
        else:
            H, G = m["heads"], m["kv_heads"]
            q, k, v = (split(lambda z, c=W.uniform(p + n + ".conv", -0.5, 0.5, d * 128, 4): _short_convolution(z, c), lin(n, d * 128)).view(-1, d, 128)
                       for n, d in (("q", G), ("k", G), ("v", H)))
            unit = lambda z: (z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 1)
            g = torch.exp(-torch.exp(W.uniform(p + "A_log", -3.0, 0.5, H)) * torch.nn.functional.softplus(lin("a", H) + W.uniform(p + "dt_bias", -2.0, 1.0, H), threshold=50.0))
            o = split(_delta, unit(q) * 128 ** -0.5, unit(k), v, g, sig(lin("b", H)))
            x = x + lin("o", w, _rms(o).reshape(-1, H * 128) * silu(lin("g", H * 128)))
        y, p = dyt(x, f"l{i}.norm2"), f"l{i}.mlp."
        x = x + lin("down", w, torch.nn.functional.gelu(lin("gate", s["ff"]), approximate="tanh") * lin("up", s["ff"]))
    return dyt(x[wanted], "final.norm") @ W.matrix("head", VOCAB, w).T


def _decayed_sum(q, k, v, decay):
    """S <- diag(decay) S + k v^T, o = S^T q, token by token for all heads of one sequence; decay [T, H, D or 1]."""
    T, H, D = q.shape
    S, out = torch.zeros(H, D, v.shape[2], dtype=v.dtype, device=v.device), torch.empty_like(v)
    for t in range(T):
        S *= decay[t, :, :, None]
        S += k[t, :, :, None] * v[t, :, None, :]
        out[t] = torch.matmul(q[t, :, None, :], S)[:, 0]
    return out


def _exact_fipitar(case, W, tokens, lengths, wanted):
    s, cfg = FIPITAR_SIZES[case["size"]], config_of(case)
    w, silu, sig, softplus = s["width"], torch.nn.functional.silu, torch.sigmoid, lambda z: torch.nn.functional.softplus(z, threshold=50.0)
    x = W.matrix("embed", VOCAB, w)[tokens]
    split = lambda f, *ts: torch.cat([f(*t) for t in zip(*(t.split(lengths) for t in ts))])
    for i, layer in enumerate(cfg["layers"]):
        p, m, kind = f"l{i}.mix.", layer["mixer"], layer["type"]
        lin = lambda n, rows, z=None: (x if z is None else z) @ W.matrix(p + n, rows, (x if z is None else z).shape[1]).T
        if kind == "gla":
            H = m["heads"]
            q, k, v = (lin(n, H * 128).view(-1, H, 128) for n in ("q", "k", "v"))
            decay = sig(lin("a2", H * 128, lin("a1", 64)) + W.matrix(p + "a2.b", H * 128)) ** (1.0 / m["tau"])
            o = split(_decayed_sum, q * 128 ** -0.5, k, v, decay.view(-1, H, 128))
            y = lin("o", w, _rms(o).reshape(-1, H * 128) * silu(lin("g", H * 128)))
        elif kind == "latent_attention":
            H, R = m["heads"], m["kv_rank"]
            q = lin("uq", H * 192, _rms(lin("dq", m["q_rank"]))).view(-1, H, 192)
            low = lin("dkv", R + 64)
            c, turned = _rms(low[:, :R]), split(lambda z: _rotate(z, m["rot"], True), low[:, None, R:])
            q = torch.cat([q[..., :128], split(lambda z: _rotate(z, m["rot"], True), q[..., 128:])], -1)
            k = torch.cat([lin("uk", H * 128, c).view(-1, H, 128), turned.expand(-1, H, -1)], -1)
            v, sink = lin("uv", H * 128, c).view(-1, H, 128), W.matrix(p + "sink", H)
            y = lin("o", w, split(lambda q, k, v: _attend(q, k, v, m["scale"], sink=sink), q, k, v))
        else:
            a, b, left = m["left"], m["right"], "left."
            H, G = a["heads"], a["kv_heads"]
            q, k, v = (lin(left + n, d * 128).view(-1, d, 128) for n, d in (("q", H), ("k", G), ("v", G)))
            zero = torch.zeros(H, dtype=torch.float64, device="cuda")
            o = split(lambda q, k, v: _attend(_rotate(_rms(q), a["rot"]), _rotate(_rms(k), a["rot"]), v, a["scale"], softcap=a["softcap"], sink=zero), q, k, v)
            y = m["left_scale"] * lin("left.o", w, (o.view(-1, H, 128) * sig(lin("left.g", H))[..., None]).reshape(-1, H * 128))
            H, V, N, G = b["heads"], b["vdim"], b["state"], b["groups"]
            inner = H * V
            proj = lin("right.in", 2 * inner + 2 * G * N + H)
            z, mixed, dt = proj.split([inner, inner + 2 * G * N, H], 1)
            weight, bias = W.uniform(p + "right.conv", -0.5, 0.5, inner + 2 * G * N, 4), W.matrix(p + "right.conv.b", inner + 2 * G * N)
            mixed = split(lambda z: _short_convolution(z, weight, bias), mixed.contiguous())
            v, k, q = mixed[:, :inner].reshape(-1, H, V), mixed[:, inner:inner + G * N].reshape(-1, G, N), mixed[:, inner + G * N:].reshape(-1, G, N)
            dt = softplus(dt + W.uniform(p + "right.dt_bias", -2.0, 1.0, H))
            decay = torch.exp(-torch.exp(W.uniform(p + "right.A_log", -3.0, 0.5, H)) * dt)
            heads = lambda t: t.repeat_interleave(H // G, 1)
            o = split(_decayed_sum, heads(q), heads(k) * dt[..., None], v, decay[..., None]) + v
            o = _rms((o.reshape(-1, inner) * silu(z)).view(-1, b["norm_groups"], inner // b["norm_groups"])).reshape(-1, inner)
            y = y + m["right_scale"] * lin("right.o", w, o)
        x = x + _layer_norm(y, W.matrix(f"l{i}.norm1.b", w))
        p = f"l{i}.mlp."
        gate, up = lin("gate", s["ff"]).clamp(max=7.0), lin("up", s["ff"]).clamp(-7.0, 7.0)
        x = x + _layer_norm(lin("down", w, gate * sig(1.702 * gate) * (up + 1.0)), W.matrix(f"l{i}.norm2.b", w))
    return _layer_norm(x[wanted], W.matrix("final.norm.b", w)) @ W.matrix("head", VOCAB, w).T


def exact(case, seed):
    """The logits of a state's first pass."""
    prompts, decoded, arriving = tokens_of(case, seed)
    steps = {"prompt": 0, "decode": 1, "serve": case["portions"]}[case["kind"]]
    sequences = [p + [decoded[k][i] for k in range(steps)] for i, p in enumerate(prompts)]
    wanted, at = [], []
    for q in sequences:
        at.append(sum(map(len, sequences[:len(at)])))
    last = [a + len(q) - 1 for a, q in zip(at, sequences)]
    if case["kind"] == "serve":
        for k in range(steps):
            wanted += [n - (steps - 1 - k) for n in last]
        wanted.append(sum(map(len, sequences)) + len(arriving) - 1)
        sequences.append(arriving)
    else:
        wanted = last
    tokens = torch.tensor([t for q in sequences for t in q], device="cuda")
    f = {"mistral": _exact_mistral, "bugidra": _exact_bugidra, "fipitar": _exact_fipitar}[case["design"]]
    with torch.no_grad():
        logits = f(case, _Weights(case, seed), tokens, [len(q) for q in sequences], torch.tensor(wanted, device="cuda"))
    if case["kind"] != "serve":
        return logits
    b = case["batch"]
    return [logits[k * b:(k + 1) * b + (k == steps - 1)] for k in range(steps)]
