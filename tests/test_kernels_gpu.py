"""Each kernel alone against a plain torch reference of the same op, at other sizes than the
engine tests use (among them the 7B model's).  The tuned bf16 kernels are also compared with
their plain kernels."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def ops():
    from flambeau_amd.kernels import ops as o
    return o


def tuned():
    from flambeau_amd.kernels import tuned as t
    return t


def rnd(*shape, dtype=torch.float32, scale=1.0, seed=0):
    g = torch.Generator(device="cpu").manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype).to(DEV)


# ---------------------------------------------------------------- element-wise and norm kernels
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V,H,n", [(300, 80, 7), (32768, 4096, 33), (5, 3, 1)])
def test_embed(dtype, V, H, n):
    table = rnd(V, H, dtype=dtype)
    tokens = torch.randint(0, V, (n,), dtype=torch.int32, device=DEV)
    out = torch.empty(n, H, dtype=torch.float32, device=DEV)
    ops().embed(table, tokens, out)
    assert torch.equal(out, table[tokens.long()].float())


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,H,eps", [(5, 96, 1e-6), (3, 4096, 1e-5), (17, 250, 1e-2), (2, 5120, 1e-5)])
def test_rmsnorm_variants(out_dtype, n, H, eps):
    x = rnd(n, H, seed=1)
    d = rnd(n, H, seed=2, scale=0.3)
    w = 1 + 0.1 * rnd(H, seed=3)
    tol = 1e-5 if out_dtype == torch.float32 else 1e-2

    def ref(v):
        v = v.double()
        return (v / torch.sqrt((v * v).mean(-1, keepdim=True) + eps) * w.double())

    out = torch.empty(n, H, dtype=out_dtype, device=DEV)
    ops().rmsnorm(x, w, out, eps)
    assert (out.double() - ref(x)).abs().max() < tol * ref(x).abs().max()
    # with the pending delta added and stored back
    x2 = x.clone()
    ops().rmsnorm(x2, w, out, eps, delta=d, store_sum=True)
    assert torch.equal(x2, x + d)
    assert (out.double() - ref(x + d)).abs().max() < tol * ref(x + d).abs().max()
    # gathered rows, nothing stored
    rows = torch.tensor([n - 1, 0, n // 2], dtype=torch.int32, device=DEV)
    out3 = torch.empty(3, H, dtype=out_dtype, device=DEV)
    x3 = x.clone()
    ops().rmsnorm(x3, w, out3, eps, delta=d, rows=rows)
    assert torch.equal(x3, x)
    assert (out3.double() - ref(x + d)[rows.long()]).abs().max() < tol * ref(x + d).abs().max()


def test_add_and_silu_mul():
    x, d = rnd(37, 1000, seed=4), rnd(37, 1000, seed=5)
    want = x + d
    ops().add_inplace(x, d)
    assert torch.equal(x, want)
    for n, I in [(3, 224), (9, 14336), (1, 5)]:
        gu = rnd(n, 2 * I, seed=6, scale=3.0)
        ref = (gu[:, :I].double() / (1 + torch.exp(-gu[:, :I].double()))) * gu[:, I:].double()
        o32 = torch.empty(n, I, dtype=torch.float32, device=DEV)
        ops().silu_mul(gu, o32)
        assert torch.allclose(o32.double(), ref, rtol=2e-6, atol=1e-6)     # float32 rounding of values up to 100
        o16 = torch.empty(n, I, dtype=torch.bfloat16, device=DEV)
        ops().silu_mul(gu, o16)
        assert (o16.double() - ref).abs().max() < 1e-2 * ref.abs().max()


# ---------------------------------------------------------------- matrix products
@pytest.mark.parametrize("M,N,K", [(1, 64, 64), (7, 100, 36), (65, 130, 250), (33, 384, 96), (2, 6144, 4096)])
def test_gemm_plain_float32(M, N, K):
    x, w = rnd(M, K, seed=7), rnd(N, K, seed=8)
    out = torch.empty(M, N, dtype=torch.float32, device=DEV)
    ops().gemm_plain(x, w, out)
    ref = x.double() @ w.double().T
    assert (out.double() - ref).abs().max() < 2e-6 * math.sqrt(K) * ref.abs().max().clamp(min=1)


def test_gemm_plain_rows_do_not_depend_on_the_batch():
    x, w = rnd(70, 300, seed=9), rnd(200, 300, seed=10)
    full = torch.empty(70, 200, dtype=torch.float32, device=DEV)
    ops().gemm_plain(x, w, full)
    one = torch.empty(1, 200, dtype=torch.float32, device=DEV)
    ops().gemm_plain(x[41:42].contiguous(), w, one)
    assert torch.equal(one[0], full[41])


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (8, 6144, 4096), (1, 4096, 14336), (64, 1024, 512),
                                   (3, 100, 72), (17, 250, 40), (5, 16, 8), (33, 28672, 4096), (1, 32768, 4096),
                                   (16, 37, 264), (49, 300, 80)])
def test_gemm_skinny_against_plain(out_dtype, M, N, K):
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=11), rnd(N, K, dtype=torch.bfloat16, seed=12, scale=0.05)
    from flambeau_amd.kernels.packing import pack_weight, unpack_weight
    packed = pack_weight(w)
    assert torch.equal(unpack_weight(packed, N, K), w)
    got = torch.full((M, N), float("nan"), dtype=out_dtype, device=DEV)
    tuned().gemm_skinny(x, packed, got)
    ref = x.double() @ w.double().T
    plain = torch.empty(M, N, dtype=out_dtype, device=DEV)
    ops().gemm_plain(x, w, plain)
    scale = ref.abs().max()
    tol = 1e-5 if out_dtype == torch.float32 else 5e-3
    assert (got.double() - ref).abs().max() < tol * scale
    assert (got.double() - plain.double()).abs().max() < 2 * tol * scale


@pytest.mark.parametrize("M,N,K", [(1, 80, 96), (7, 48, 1024), (5, 37, 264), (16, 6144, 512), (12, 4112, 72), (9, 16400, 2560), (8, 4096, 14336),
                                   (12, 1024, 4096), (6, 1024, 4096)])
def test_gemm_skinny_with_several_row_groups_per_block(M, N, K):
    """One or two row groups per block (the last block may hold one), x fetched piece by piece or by
    rows through LDS, and any number of waves give the same numbers as long as K is split over the
    same number of waves; plain and SwiGLU epilogue."""
    from flambeau_amd.kernels.packing import pack_weight
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=13), rnd(N, K, dtype=torch.bfloat16, seed=14, scale=0.05)
    packed = pack_weight(w)
    ref = x.double() @ w.double().T
    for waves in (0, 2, 4, 8, 16):                    # 0: the kernel's own choice
        outs = []
        for groups in (1, 2):
            for direct_x in (0, 1):
                got = torch.full((M, N), float("nan"), dtype=torch.float32, device=DEV)
                tuned().gemm_skinny(x, packed, got, waves + 256 * groups + 65536 * direct_x)
                assert (got.double() - ref).abs().max() < 1e-5 * ref.abs().max()
                outs.append(got)
        if waves in (2, 4, 8) and K // 32 >= 2 * waves:       # (fewer steps than that: the kernel takes fewer waves)
            assert all(torch.equal(outs[0], o) for o in outs[1:])
    if N % 32 == 0:
        gate, up = w[:N // 2].contiguous(), w[N // 2:].contiguous()
        Wgu = tuned().prepare_gate_up(gate, up)
        gr, ur = x.double() @ gate.double().T, x.double() @ up.double().T
        ref_act = gr / (1 + torch.exp(-gr)) * ur
        for groups in (1, 2):
            act = torch.full((M, N // 2), float("nan"), dtype=torch.float32, device=DEV)
            tuned().gemm_skinny(x, Wgu.packed, act, 256 * groups, swiglu_rows=Wgu.packed_rows)
            assert (act.double() - ref_act).abs().max() < 1e-5 * ref_act.abs().max()
    with pytest.raises(Exception, match="row groups"):
        tuned().gemm_skinny(x, packed, torch.empty(M, N, dtype=torch.float32, device=DEV), 256 * 3)


@pytest.mark.parametrize("M,H,N2,I,eps", [(1, 4096, 6144, 512, 1e-5), (8, 4096, 32768, 14336, 1e-5), (16, 72, 40, 104, 1e-2),
                                            (8, 5104, 6144, 96, 1e-5), (12, 5120, 28672, 256, 1e-5),
                                            (3, 136, 250, 40, 1e-6), (5, 64, 16, 8, 1e-5),
                                            (64, 4096, 6144, 14336, 1e-5), (17, 96, 40, 64, 1e-3), (40, 2080, 300, 160, 1e-5),
                                            (2048, 4096, 1024, 512, 1e-5), (300, 264, 152, 96, 1e-6), (129, 72, 40, 104, 1e-3),
                                            (128, 4096, 6144, 4096, 1e-5), (100, 520, 64, 2048, 1e-5), (512, 5120, 256, 1024, 1e-5)])
def test_gemm_fused_with_the_norms_around_it(M, H, N2, I, eps):
    from flambeau_amd.kernels import KernelError
    """resid += a W1^T in the product's epilogue, norm(resid) W2^T through the row scale of the next
    product, against the same chain in float64; and the SwiGLU epilogue after a row scale.  Up to 16
    rows in the skinny kernel, 17 to 64 in the kernel that shares x through LDS, more in the tiled one."""
    from flambeau_amd.kernels.packing import pack_weight
    a = rnd(M, I, dtype=torch.bfloat16, seed=51)
    w1 = rnd(H, I, dtype=torch.bfloat16, seed=52, scale=0.05)
    w2 = rnd(N2, H, dtype=torch.bfloat16, seed=53, scale=0.05)
    g = rnd(H, seed=54).abs() + 0.5
    resid0 = rnd(M, H, seed=55)
    resid = resid0.clone()
    xg = torch.full((M, H), float("nan"), dtype=torch.bfloat16, device=DEV)
    if M <= 16:
        ssq = torch.full((M, tuned().skinny_parts(H)), float("nan"), dtype=torch.float32, device=DEV)
        rows = tuned().gemm_skinny_residual(a, pack_weight(w1), resid, g, xg, ssq, eps)
    elif M <= 64:
        ssq = torch.full((M, tuned().mid_parts(H)), float("nan"), dtype=torch.float32, device=DEV)
        ws = torch.full((tuned().gemm_mid_splits(M, H, I) * M * H,), float("nan"), dtype=torch.float32, device=DEV)
        rows = tuned().gemm_mid_residual(a, pack_weight(w1), resid, g, xg, ssq, eps, ws)
    else:
        splits = tuned().gemm_tiled_splits(M, H, I)
        ws = torch.full((splits * M * H,), float("nan"), dtype=torch.float32, device=DEV) if splits > 1 else None
        if splits > 1:
            with pytest.raises(KernelError, match="workspace"):
                tuned().gemm_tiled_residual(a, pack_weight(w1), resid, g, xg, torch.empty(M, tuned().tiled_parts(M, H, I), device=DEV), eps)
        ssq = torch.full((M, tuned().tiled_parts(M, H, I)), float("nan"), dtype=torch.float32, device=DEV)
        rows = tuned().gemm_tiled_residual(a, pack_weight(w1), resid, g, xg, ssq, eps, ws)
    r_ref = resid0.double() + a.double() @ w1.double().T
    assert (resid.double() - r_ref).abs().max() < 1e-5 * r_ref.abs().max()
    assert (ssq.double().sum(1) - (r_ref ** 2).sum(1)).abs().max() < 1e-5 * (r_ref ** 2).sum(1).max()
    assert (xg.double() - r_ref * g.double()).abs().max() < 5e-3 * (r_ref * g.double()).abs().max()
    normed = r_ref * torch.rsqrt((r_ref ** 2).mean(1, keepdim=True) + eps) * g.double()
    ref = normed @ w2.double().T
    class Rt:
        def buffer(self, name, n, cols, dtype=torch.bfloat16, max_rows=None):
            return torch.empty(n, cols, dtype=dtype, device=DEV)
    W2 = tuned().prepare_weight(w2)
    got = torch.full((M, N2), float("nan"), dtype=torch.float32, device=DEV)
    tuned().gemm(rows, W2, got, Rt())
    assert (got.double() - ref).abs().max() < 6e-3 * ref.abs().max()
    # the rows themselves, for kernels that do not take the factors
    made = rows.materialize(Rt())
    assert (made.double() - normed).abs().max() < 5e-3 * normed.abs().max()
    if N2 % 32 == 0:
        gate, up = w2[:N2 // 2].contiguous(), w2[N2 // 2:].contiguous()
        Wgu = tuned().prepare_gate_up(gate, up)
        act = torch.full((M, N2 // 2), float("nan"), dtype=torch.float32, device=DEV)
        tuned().gemm_swiglu(rows, Wgu, act, Rt())
        gr, ur = normed @ gate.double().T, normed @ up.double().T
        ref_act = gr / (1 + torch.exp(-gr)) * ur
        assert (act.double() - ref_act).abs().max() < 1e-2 * ref_act.abs().max()


def test_gemm_skinny_refuses_what_it_cannot_do():
    from flambeau_amd.kernels import KernelError
    from flambeau_amd.kernels.packing import pack_weight
    x, w = rnd(2, 36, dtype=torch.bfloat16), rnd(5, 36, dtype=torch.bfloat16)
    out = torch.empty(2, 5, dtype=torch.float32, device=DEV)
    with pytest.raises(KernelError, match="multiple of 8"):
        tuned().gemm_skinny(x, pack_weight(w), out)
    prepared = tuned().prepare_weight(w)
    assert prepared.packed is None                 # the dispatcher takes the plain kernel instead
    tuned().gemm(x, prepared, out)
    assert (out.double() - x.double() @ w.double().T).abs().max() < 1e-4
    with pytest.raises(KernelError, match="at most 64"):
        tuned().gemm_skinny(rnd(65, 64, dtype=torch.bfloat16), pack_weight(rnd(8, 64, dtype=torch.bfloat16)),
                            torch.empty(65, 8, dtype=torch.float32, device=DEV))
    with pytest.raises(KernelError, match="packs to"):
        tuned().gemm_skinny(rnd(2, 64, dtype=torch.bfloat16), pack_weight(rnd(8, 32, dtype=torch.bfloat16)), out)
    with pytest.raises(KernelError, match="at most 16 rows"):       # the fusions with the norm: one tile of tokens
        tuned().gemm_skinny_residual(rnd(17, 64, dtype=torch.bfloat16), pack_weight(rnd(32, 64, dtype=torch.bfloat16)),
                                     rnd(17, 32), rnd(32), torch.empty(17, 32, dtype=torch.bfloat16, device=DEV),
                                     torch.empty(17, 2, dtype=torch.float32, device=DEV), 1e-5)


# ---------------------------------------------------------------- cache, rotation, attention
def make_cache(n_pages, nkv, ps, hd, dtype):
    from flambeau_amd.kernels.ops import PagedLayerCache
    return PagedLayerCache(torch.zeros(n_pages, 2, nkv, ps, hd, dtype=dtype, device=DEV))


def read_cache(cache, table_row, t, kvh):
    """Key and value rows of token t through the block table (V is stored transposed in a page)."""
    ps, hd = cache.page_size, cache.head_dim
    page, r = int(table_row[t // ps]), t % ps
    k = cache.pool[page, 0, kvh].reshape(ps, hd)[r]
    v = cache.pool[page, 1, kvh].reshape(hd, ps)[:, r]
    return k, v


def rope_ref(x, pos, theta, rot):
    """x [n, heads, hd] double."""
    half = rot // 2
    inv = theta ** (-2.0 * torch.arange(half, dtype=torch.float64, device=x.device) / rot)
    ang = pos.double()[:, None] * inv[None]
    c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    out = x.clone()
    lo, hi = x[..., :half], x[..., half:rot]
    out[..., :half] = lo * c - hi * s
    out[..., half:rot] = lo * s + hi * c
    return out


@pytest.mark.parametrize("parts", [2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("nh,nkv,hd,rot,paired", [(4, 2, 128, 128, True), (3, 1, 200, 64, False), (2, 2, 24, 0, False), (5, 1, 16, 16, True)])
def test_rope_kv_write_adds_parts_in_order(nh, nkv, hd, rot, paired, parts):
    """Partial sums, whatever their number and the heads' size: the bits of their sum in rising order."""
    n, ps = 21, 16
    cache, again = make_cache(8, nkv, ps, hd, torch.bfloat16), make_cache(8, nkv, ps, hd, torch.bfloat16)
    pos = torch.arange(n, dtype=torch.int32, device=DEV)
    seq = torch.zeros(n, dtype=torch.int32, device=DEV)
    table = torch.tensor([[5, 2]], dtype=torch.int32, device=DEV)
    qkv = rnd(parts, n, (nh + 2 * nkv) * hd, seed=parts)
    whole = qkv[0].clone()
    for part in qkv[1:]:
        whole += part
    outs = [torch.zeros(n, nh * hd, dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    ops().rope_kv_write(qkv, pos, seq, table, outs[0], cache, nh, rot, 1e4, paired=paired, parts=parts)
    ops().rope_kv_write(whole, pos, seq, table, outs[1], again, nh, rot, 1e4, paired=paired)
    live = [5, 2]
    assert torch.equal(outs[0], outs[1]) and torch.equal(cache.pool[live].nan_to_num(), again.pool[live].nan_to_num())


@pytest.mark.parametrize("nh,nkv,hd,rot", [(8, 2, 256, 64), (32, 8, 128, 64)])
def test_rope_kv_write_reads_the_parts_there_are_and_no_more(nh, nkv, hd, rot):
    """Two parts are one read more per value: measured 1.03 to 1.06 of one part's time, and 1.15 to 1.21 where four reads are asked for whatever there is."""
    n, ps = 2048, 16
    cache = make_cache(n // ps, nkv, ps, hd, torch.bfloat16)
    pos, seq = torch.arange(n, dtype=torch.int32, device=DEV), torch.zeros(n, dtype=torch.int32, device=DEV)
    table = torch.arange(n // ps, dtype=torch.int32, device=DEV).view(1, -1)
    qkv, out = rnd(2, n, (nh + 2 * nkv) * hd, seed=3), torch.zeros(n, nh * hd, dtype=torch.bfloat16, device=DEV)
    times = times_in_turn(*(lambda p=p: ops().rope_kv_write(qkv if p == 2 else qkv[0], pos, seq, table, out, cache, nh, rot, 1e4, parts=p) for p in (1, 2)))
    assert times[1] < 1.12 * times[0], times


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,hd,ps,rot,theta", [(4, 2, 16, 8, 16, 1e4), (6, 1, 24, 16, 24, 1e6),
                                                   (32, 8, 128, 16, 128, 1e6), (3, 3, 40, 4, 20, 5e5),
                                                   (2, 1, 64, 32, 0, 1.0)])
def test_rope_kv_write(dtype, nh, nkv, hd, ps, rot, theta):
    seqs = [(0, 5), (37, 3), (ps - 1, 2), (100, 1)]          # (start position, tokens)
    n = sum(q for _, q in seqs)
    n_pages = 96
    cache = make_cache(n_pages, nkv, ps, hd, dtype)
    perm = torch.randperm(n_pages)
    table = torch.full((len(seqs), 56), -1, dtype=torch.int32)
    used = 0
    pos, tok_seq = [], []
    for s, (st, q) in enumerate(seqs):
        nb = -(-(st + q) // ps)
        table[s, :nb] = perm[used:used + nb].int()
        used += nb
        pos += list(range(st, st + q))
        tok_seq += [s] * q
    pos_d = torch.tensor(pos, dtype=torch.int32, device=DEV)
    seq_d = torch.tensor(tok_seq, dtype=torch.int32, device=DEV)
    qkv = rnd(n, (nh + 2 * nkv) * hd, seed=13)
    q_out = torch.empty(n, nh * hd, dtype=dtype, device=DEV)
    ops().rope_kv_write(qkv, pos_d, seq_d, table.to(DEV), q_out, cache, nh, rot, theta)
    x = qkv.double()
    q_ref = x[:, :nh * hd].reshape(n, nh, hd)
    k_ref = x[:, nh * hd:(nh + nkv) * hd].reshape(n, nkv, hd)
    v_ref = x[:, (nh + nkv) * hd:].reshape(n, nkv, hd)
    if rot:
        q_ref, k_ref = rope_ref(q_ref, pos_d, theta, rot), rope_ref(k_ref, pos_d, theta, rot)
    tol = 2e-5 if dtype == torch.float32 else 1e-2
    assert (q_out.double().reshape(n, nh, hd) - q_ref).abs().max() < tol * 4
    for i in range(n):
        for h in range(nkv):
            k, v = read_cache(cache, table[tok_seq[i]], pos[i], h)
            assert (k.double() - k_ref[i, h]).abs().max() < tol * 4
            assert (v.double() - v_ref[i, h]).abs().max() < tol * 4
    # nothing else was touched: untouched pages are still zero
    touched = set(int(p) for p in table[table >= 0])
    for p in range(n_pages):
        if p not in touched:
            assert not cache.pool[p].any()
    # the same with the angles from the step's table, and with the projection's rows in paired order
    from flambeau_amd.kernels.packing import rotary_paired_rows
    variants = []
    if rot:
        angles = torch.full((n, rot // 2, 2), float("nan"), dtype=torch.float32, device=DEV)
        ops().rope_table(pos_d, rot, theta, angles)
        variants.append(dict(table=angles))
        order = rotary_paired_rows(nh, nkv, hd, rot)
        assert (order is None) == bool(rot % 16 or hd % 16)
        if order is not None:
            assert sorted(order.tolist()) == list(range((nh + 2 * nkv) * hd))
            variants.append(dict(table=angles, paired=True, order=order))
    for v in variants:
        cache2 = make_cache(n_pages, nkv, ps, hd, dtype)
        q2 = torch.empty_like(q_out)
        order = v.pop("order", None)
        src = qkv if order is None else qkv[:, order.to(DEV)].contiguous()
        ops().rope_kv_write(src, pos_d, seq_d, table.to(DEV), q2, cache2, nh, rot, theta, **v)
        assert torch.equal(q2, q_out) and torch.equal(cache2.pool, cache.pool)


def attention_ref(q, keys, vals, pos, scale, window):
    """One query row per call site: q [nh, hd], keys/vals [T, nkv, hd] double, query at ``pos``."""
    nh, nkv = q.shape[0], keys.shape[1]
    lo = max(0, pos - window + 1) if window else 0
    out = torch.zeros_like(q)
    for h in range(nh):
        g = h // (nh // nkv)
        s = (keys[lo:pos + 1, g] @ q[h]) * scale
        p = torch.softmax(s, 0)
        out[h] = p @ vals[lo:pos + 1, g]
    return out


def build_attention_case(dtype, nh, nkv, hd, ps, seqs, seed=0):
    """Random cache contents for requests ``seqs`` = (context length, query length); the queries
    are the last ``q`` positions of each.  Returns what the kernels take and the reference."""
    torch.manual_seed(seed)
    n_pages = sum(-(-c // ps) for c, _ in seqs) + 3
    cache = make_cache(n_pages, nkv, ps, hd, dtype)
    perm = torch.randperm(n_pages)
    width = max(-(-c // ps) for c, _ in seqs) + 1
    table = torch.full((len(seqs), width), -1, dtype=torch.int32)
    used = 0
    K, V = [], []
    for s, (c, _) in enumerate(seqs):
        nb = -(-c // ps)
        table[s, :nb] = perm[used:used + nb].int()
        used += nb
        k = (torch.randn(c, nkv, hd) * 0.8).to(dtype)
        v = torch.randn(c, nkv, hd).to(dtype)
        K.append(k.double().to(DEV))
        V.append(v.double().to(DEV))
        for t in range(c):
            page, r = int(table[s, t // ps]), t % ps
            cache.pool[page, 0].reshape(nkv, ps, hd)[:, r] = k[t].to(DEV)
            cache.pool[page, 1].reshape(nkv, hd, ps)[:, :, r] = v[t].to(DEV)
    pos, tok_seq = [], []
    for s, (c, ql) in enumerate(seqs):
        pos += list(range(c - ql, c))
        tok_seq += [s] * ql
    n = len(pos)
    q = (torch.randn(n, nh, hd) * 0.8).to(dtype).to(DEV)
    return dict(cache=cache, table=table.to(DEV), K=K, V=V, pos=pos, tok_seq=tok_seq, q=q, n=n,
                pos_d=torch.tensor(pos, dtype=torch.int32, device=DEV),
                seq_d=torch.tensor(tok_seq, dtype=torch.int32, device=DEV))


def attention_case_ref(case, scale, window):
    outs = []
    for i in range(case["n"]):
        s = case["tok_seq"][i]
        outs.append(attention_ref(case["q"][i].double(), case["K"][s], case["V"][s], case["pos"][i], scale, window))
    return torch.stack(outs)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,hd,ps,window", [(4, 2, 16, 8, 0), (6, 1, 24, 16, 11), (8, 2, 128, 16, 0),
                                                (5, 5, 72, 4, 30), (2, 2, 256, 32, 0), (3, 1, 10, 2, 5)])
def test_attn_plain(dtype, nh, nkv, hd, ps, window):
    seqs = [(70, 70), (33, 1), (ps * 3, 2), (1, 1), (50, 9)]
    case = build_attention_case(dtype, nh, nkv, hd, ps, seqs)
    scale = 1 / math.sqrt(hd)
    out = torch.empty(case["n"], nh * hd, dtype=dtype, device=DEV)
    ops().attn_plain(case["q"].reshape(case["n"], nh * hd), out, case["cache"], case["pos_d"], case["seq_d"],
                     case["table"], nh, scale, window)
    ref = attention_case_ref(case, scale, window)
    tol = 2e-6 if dtype == torch.float32 else 1e-2
    assert (out.double().reshape(case["n"], nh, hd) - ref).abs().max() < tol * ref.abs().max()


def test_attn_plain_refuses_large_heads():
    from flambeau_amd.kernels import KernelError
    case = build_attention_case(torch.float32, 1, 1, 8, 4, [(4, 1)])
    big = make_cache(2, 1, 4, 264, torch.float32)
    with pytest.raises(KernelError, match="head size 264"):
        ops().attn_plain(torch.zeros(1, 264, device=DEV), torch.zeros(1, 264, device=DEV), big, case["pos_d"],
                         case["seq_d"], case["table"], 1, 1.0, 0)


# ---------------------------------------------------------------- sampling
@pytest.mark.parametrize("R,V", [(1, 10), (5, 384), (3, 32768), (8, 131072), (2, 257)])
def test_argmax_first_maximum_wins(R, V):
    logits = rnd(R, V, seed=14)
    logits[0, V // 3] = 50.0
    logits[0, V - 1] = 50.0            # a later tie loses
    out = torch.empty(R, dtype=torch.int32, device=DEV)
    ops().argmax(logits, out)
    want = [int(np.argmax(row)) for row in logits.cpu().numpy()]
    assert out.tolist() == want and out[0] == V // 3


@pytest.mark.parametrize("V", [97, 384, 32768])
def test_sample_is_the_inverse_cdf_in_index_order(V):
    import plain_model as pm
    R = 64
    logits = rnd(R, V, seed=15, scale=2.0)
    u = torch.rand(R, generator=torch.Generator().manual_seed(1)).to(DEV)
    u[0], u[1] = 0.0, 0.999999
    inv_t = torch.full((R,), 1 / 0.8, device=DEV)
    inv_t[2] = 0.0                                       # greedy row among the others
    out = torch.empty(R, dtype=torch.int32, device=DEV)
    ops().sample(logits, inv_t, u, out)
    l, uu = logits.cpu().double().numpy(), u.cpu().double().numpy()
    assert out[2] == int(np.argmax(l[2]))
    bad = 0
    for r in range(R):
        if r == 2:
            continue
        p = np.exp((l[r] - l[r].max()) / 0.8)
        cdf = np.cumsum(p) / p.sum()
        want = int(np.searchsorted(cdf, uu[r], side="left"))
        got = int(out[r])
        if got != want:
            # a draw within rounding of a boundary may fall to the neighbour
            assert abs(got - want) == 1 and abs(cdf[min(got, want)] - uu[r]) < 1e-5
            bad += 1
    assert bad <= 2


@pytest.mark.parametrize("V", [97, 1000, 40000])
def test_penalties_and_bias_are_the_host_sampler_s(V):
    """Penalties from per-slot token counts and the bias triples against the host's rule, bit for bit:
    rows with and without a history, neutral penalties, tokens seen several times, a slot that is
    counted anew for another request, and the counts after a draw has joined them."""
    from flambeau_amd.sampling.host import penalised
    from flambeau_amd.sampling.params import SamplingParams
    rng = np.random.default_rng(V + 1)
    n_slots, R = 7, 6
    slots = [2, -1, 0, 5, 1, 3]
    params = [SamplingParams(repetition_penalty=1.7), SamplingParams(), SamplingParams(presence_penalty=0.6, frequency_penalty=0.35),
              SamplingParams(repetition_penalty=0.8, frequency_penalty=1.25), SamplingParams(),
              SamplingParams(repetition_penalty=1.3, presence_penalty=-0.4, logit_bias={1: 2.0, V - 1: -3.5, V + 5: 9.0})]
    params[1] = SamplingParams(logit_bias={0: 1.5, 17: -0.25})
    histories = [rng.integers(0, min(V, 40), int(n)).tolist() for n in (50, 0, 9, 200, 30, 0)]
    histories[3][:3] = [V - 1, V - 1, 0]
    counts = torch.randint(0, 9, (n_slots, V), dtype=torch.int16, device=DEV)       # what other requests left behind
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    f32 = lambda v: torch.tensor(np.asarray(v, dtype=np.float32), device=DEV)
    for s, h in zip(slots, histories):
        if s >= 0:
            ops().sample_history(counts, s, i32(h))
    for s, h in zip(slots, histories):
        if s >= 0:
            assert counts[s].tolist() == np.bincount(h, minlength=V).tolist()
    assert counts[4].max() > 0 and counts[6].max() > 0                                # rows nobody took are untouched
    logits = rnd(R, V, seed=21, scale=3.0)
    want = [penalised(l, p, h) for l, p, h in zip(logits.cpu().numpy(), params, histories)]

    def apply(l):
        ops().sample_penalise(l, counts, f32(slots), f32([p.repetition_penalty for p in params]),
                              f32([p.presence_penalty for p in params]), f32([p.frequency_penalty for p in params]))
        triples = [(r, t, b) for r, p in enumerate(params) if p.logit_bias for t, b in p.logit_bias.items() if t < V]
        ops().sample_bias(l, *(f32(list(c)) for c in zip(*triples)))
        return l
    got = apply(logits.clone())
    assert torch.equal(got.cpu(), torch.tensor(np.stack(want)))
    assert not torch.equal(got[0], logits[0]) and torch.equal(got[4], logits[4])
    # the drawn tokens join the histories (a row without a slot counts nowhere; a token twice in a row adds up)
    for draw in ([3, 5, 3, V - 1, 0, 8], [3, 5, 7, V - 1, 0, 8]):
        before = counts.clone()
        ops().sample_count(counts, f32(slots), i32(draw))
        for s, h, t in zip(slots, histories, draw):
            if s >= 0:
                h.append(t)
        changed = (counts != before).nonzero().tolist()
        assert sorted(changed) == sorted([s, t] for s, t in zip(slots, draw) if s >= 0)
    want = [penalised(l, p, h) for l, p, h in zip(logits.cpu().numpy(), params, histories)]
    assert torch.equal(apply(logits.clone()).cpu(), torch.tensor(np.stack(want)))
    # counts stop at 65,535
    ops().sample_history(counts, 6, i32([4] * 3))
    counts[6, 4] = -2                                                               # 65,534 as 16 bits
    for _ in range(3):
        ops().sample_count(counts, f32([6.0]), i32([4]))
    assert int(counts[6, 4]) == -1


@pytest.mark.parametrize("V", [97, 1000, 32768, 131072])
def test_filtered_sample_is_the_host_sampler_s(V):
    """Top-k, top-p and min-p on the device against the host sampler (itself checked against the plain
    one) with the same uniform numbers: rows of every combination of filters, logits with ties, rows
    without a filter and greedy rows among them (those keep what the plain kernel drew)."""
    from flambeau_amd.sampling.host import sample_host
    from flambeau_amd.sampling.params import SamplingParams
    rng = np.random.default_rng(V)
    combos = []
    for top_k in (None, 1, 5, 40, 700, 2048):
        for top_p in (None, 0.15, 0.9, 0.999, 1.0):
            for min_p in (None, 0.02, 0.6):
                combos.append((top_k, top_p, min_p))
    R = len(combos) + 2
    logits = rnd(R, V, seed=16, scale=2.5)
    logits[3] = torch.round(logits[3] * 2) / 2            # many equal logits: ties go by index
    logits[7, :] = 0.25                                    # all equal
    logits[9] = torch.round(logits[9])
    temps = rng.choice([0.6, 0.8, 1.0, 1.7], R).tolist()
    us = rng.random(R).astype(np.float32)
    us[4], us[5] = 0.0, np.float32(0.9999999)
    params = [SamplingParams(temperature=t, top_k=c[0], top_p=c[1], min_p=c[2]) for t, c in zip(temps, combos)]
    params += [SamplingParams(temperature=0.9), SamplingParams(temperature=0.0, top_k=5)]       # no filter; greedy
    assert all(p.device_ok for p in params)
    f32 = lambda v: torch.tensor(np.asarray(v, dtype=np.float32), device=DEV)
    inv_t = f32([0.0 if p.is_greedy else 1.0 / p.temperature for p in params])
    filt = [p.device_filters for p in params]
    out = torch.full((R,), -1, dtype=torch.int32, device=DEV)
    plain_draw = torch.empty(R, dtype=torch.int32, device=DEV)
    ops().sample(logits, inv_t, f32(us), plain_draw)
    out.copy_(plain_draw)
    args = (logits, inv_t, f32(us), f32([f[0] for f in filt]), f32([f[1] for f in filt]), f32([f[2] for f in filt]))
    ops().sample_filtered(*args, out)
    if V > 32768:
        # with scratch for the probabilities (formed once instead of in every pass): the same draws
        again = plain_draw.clone()
        ops().sample_filtered(*args, again, stash=torch.empty(R * V, dtype=torch.int32, device=DEV))
        assert torch.equal(again, out)
    assert out[R - 2] == plain_draw[R - 2] and out[R - 1] == plain_draw[R - 1] == int(torch.argmax(logits[R - 1]))

    class OneNumber:
        def __init__(self, u): self.u = u
        def next_f32(self): return self.u
    l = logits.cpu().numpy()
    differ = 0
    for r in range(R - 2):
        want = sample_host(l[r], params[r], [], OneNumber(us[r]))
        got = int(out[r])
        if got != want:
            # sums in another order: a draw on a boundary may fall to the neighbour in the order of probability
            p = np.exp((l[r].astype(np.float64) - l[r].max()) / temps[r]); p /= p.sum()
            order = np.argsort(-p, kind="stable").tolist()
            assert abs(order.index(got) - order.index(want)) == 1, (r, combos[r], got, want)
            differ += 1
    assert differ <= 2
    # a filter that leaves one candidate is the argmax, whatever the number drawn
    for r, c in enumerate(combos):
        if c[0] == 1:
            assert int(out[r]) == int(np.argmax(l[r]))


# ---------------------------------------------------------------- tuned attention for single rows
def decode_rows(case, picked):
    """(row, position, request, 0) of the picked rows, as the decode kernel wants them."""
    pos, seq = case["pos_d"].cpu().tolist(), case["seq_d"].cpu().tolist()
    return torch.tensor([[r, pos[r], seq[r], 0] for r in picked], dtype=torch.int32, device=DEV).reshape(-1, 4)


@pytest.mark.parametrize("n_split", [1, 2, 5])
@pytest.mark.parametrize("nh,nkv,hd,ps,window", [(32, 8, 128, 16, 0), (4, 2, 16, 8, 16), (6, 1, 24, 16, 0),
                                                (5, 5, 32, 16, 24), (20, 1, 64, 8, 0), (8, 4, 256, 32, 100),
                                                (3, 1, 40, 64, 0)])
def test_attn_decode_against_plain_and_reference(nh, nkv, hd, ps, window, n_split):
    seqs = [(700, 1), (33, 1), (ps * 3, 1), (1, 1), (257, 3), (64, 2), (32, 1), (31, 1)]
    case = build_attention_case(torch.bfloat16, nh, nkv, hd, ps, seqs, seed=3)
    n = case["n"]
    scale = 1 / math.sqrt(hd)
    q2 = case["q"].reshape(n, nh * hd)
    rows = decode_rows(case, reversed(range(n)))      # any order of rows
    out = torch.full((n, nh * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    hdp = -(-hd // 32) * 32
    part_o = torch.empty(n * nh * n_split * hdp, dtype=torch.float32, device=DEV)
    part_ml = torch.empty(n * nh * n_split * 2, dtype=torch.float32, device=DEV)
    tuned().attn_decode(q2, out, case["cache"], rows, case["table"], nh, scale, window, n_split, part_o, part_ml)
    plain = torch.empty_like(out)
    ops().attn_plain(q2, plain, case["cache"], case["pos_d"], case["seq_d"], case["table"], nh, scale, window)
    ref = attention_case_ref(case, scale, window)
    top = ref.abs().max()
    assert (out.double().reshape(n, nh, hd) - ref).abs().max() < 1e-2 * top
    assert (out.double() - plain.double()).abs().max() < 1.5e-2 * top


@pytest.mark.parametrize("nh,nkv,hd,ps,window", [(32, 8, 128, 16, 0), (4, 2, 16, 8, 16), (6, 1, 24, 16, 0), (20, 1, 64, 8, 0),
                                                (8, 4, 256, 32, 100), (40, 2, 32, 16, 0)])
def test_attn_decode_with_splits_per_row(nh, nkv, hd, ps, window):
    """Rows with splits of their own (long contexts many, short ones one, unused places in the list):
    the reference's result, and exactly the uniform kernel's where a row has one split."""
    seqs = [(1500, 1), (33, 1), (ps * 3, 1), (1, 1), (257, 3), (640, 2), (32, 1), (31, 1)]
    case = build_attention_case(torch.bfloat16, nh, nkv, hd, ps, seqs, seed=9)
    n = case["n"]
    scale = 1 / math.sqrt(hd)
    q2 = case["q"].reshape(n, nh * hd)
    rows = decode_rows(case, range(n))
    per_row = tuned().decode_blocks_per_row(nh, nkv)
    items_host, firsts_host = tuned().balanced_items(rows.cpu().numpy(), per_row, window)
    splits = {int(r): int(w) >> 8 for r, _, _, w in items_host if r >= 0}
    assert len(items_host) == tuned().decode_item_budget(n, per_row) and set(splits) == set(range(n))
    assert (max(splits.values()) > 1 or 0 < window < 256) and min(splits.values()) == 1
    assert (items_host[:, 0] < 0).any() == (sum(splits.values()) < len(items_host))
    items, firsts = torch.tensor(items_host, device=DEV), torch.tensor(firsts_host, device=DEV)
    assert all(items_host[f, 0] == r and items_host[f, 3] == 256 * k for r, f, k, _ in firsts_host)
    hdp = -(-hd // 32) * 32
    part_o = torch.full((len(items_host) * nh * hdp,), float("nan"), dtype=torch.float32, device=DEV)
    part_ml = torch.full((len(items_host) * nh * 2,), float("nan"), dtype=torch.float32, device=DEV)
    out = torch.full((n, nh * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    tuned().attn_decode(q2, out, case["cache"], items, case["table"], nh, scale, window, 0, part_o, part_ml, firsts=firsts)
    ref = attention_case_ref(case, scale, window)
    assert (out.double().reshape(n, nh, hd) - ref).abs().max() < 1e-2 * ref.abs().max()
    whole = torch.empty_like(out)
    tuned().attn_decode(q2, whole, case["cache"], rows, case["table"], nh, scale, window, 1)
    one = [r for r, k in splits.items() if k == 1]
    assert torch.equal(out[one], whole[one])
    # a list with a place per row: nothing to merge, no workspace
    plain_items = rows.clone()
    plain_items[:, 3] = 256
    again = torch.full_like(out, float("nan"))
    tuned().attn_decode(q2, again, case["cache"], plain_items, case["table"], nh, scale, window, 0)
    assert torch.equal(again, whole)


def test_attn_decode_subset_of_rows_leaves_the_others_alone():
    nh, nkv, hd, ps = 8, 2, 64, 16
    case = build_attention_case(torch.bfloat16, nh, nkv, hd, ps, [(40, 4), (90, 1)], seed=4)
    n = case["n"]
    q2 = case["q"].reshape(n, nh * hd)
    out = torch.full((n, nh * hd), 7.0, dtype=torch.bfloat16, device=DEV)
    tuned().attn_decode(q2, out, case["cache"], decode_rows(case, [4, 1]), case["table"], nh, 0.125, 0, 1)
    ref = attention_case_ref(case, 0.125, 0)
    assert (out[[0, 2, 3]] == 7.0).all()
    assert (out[[1, 4]].double().reshape(2, nh, hd) - ref[[1, 4]]).abs().max() < 1e-2 * ref.abs().max()


def test_attn_decode_takes_more_items_than_a_grid_has_places():
    """70,000 single rows in one call (the grid's slow index holds 65,535): all of them are computed,
    in the uniform form with two splits and with a list of items."""
    nh, nkv, hd, ps, n = 2, 1, 16, 8, 70000
    case = build_attention_case(torch.bfloat16, nh, nkv, hd, ps, [(40, 1), (23, 1)], seed=2)
    q = (torch.randn(n, nh, hd, generator=torch.Generator().manual_seed(3)) * 0.8).to(torch.bfloat16).to(DEV)
    req = torch.arange(n, device=DEV) % 2
    pos = torch.where(req == 0, torch.arange(n, device=DEV) % 40, torch.arange(n, device=DEV) % 23)
    rows = torch.stack([torch.arange(n, device=DEV), pos, req, torch.zeros_like(req)], 1).int().contiguous()
    # the reference, all rows at once: scores against every key of the row's request, masked beyond its position
    ref = torch.zeros(n, nh, hd, dtype=torch.float64, device=DEV)
    for r in range(2):
        sel = (req == r).nonzero().squeeze(1)
        K, V = case["K"][r][:, 0], case["V"][r][:, 0]
        s = torch.einsum("nhd,td->nht", q[sel].double(), K) * 0.25
        s = s.masked_fill(torch.arange(K.shape[0], device=DEV)[None, None, :] > pos[sel][:, None, None], float("-inf"))
        ref[sel] = torch.einsum("nht,td->nhd", torch.softmax(s, -1), V)
    hdp = 32
    for n_split in (2, 0):
        out = torch.full((n, nh * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
        items = rows.clone()
        k = max(n_split, 1)
        if n_split == 0:
            items[:, 3] = 256
        part_o = torch.empty(n * nh * k * hdp, dtype=torch.float32, device=DEV)
        part_ml = torch.empty(n * nh * k * 2, dtype=torch.float32, device=DEV)
        tuned().attn_decode(q.reshape(n, nh * hd), out, case["cache"], items, case["table"], nh, 0.25, 0, n_split, part_o, part_ml)
        err = (out.double().reshape(n, nh, hd) - ref).abs().amax((1, 2))
        assert not torch.isnan(out).any() and err.max() < 1e-2 * ref.abs().max(), int(err.argmax())


# ---------------------------------------------------------------- tiled matrix product
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(128, 128, 64), (65, 100, 72), (300, 250, 40), (2048, 512, 256), (129, 37, 264),
                                   (70, 4096, 4096), (200, 6144, 512), (513, 384, 96), (1000, 130, 1000)])
def test_gemm_tiled_against_plain(out_dtype, M, N, K):
    from flambeau_amd.kernels.packing import pack_weight
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=21), rnd(N, K, dtype=torch.bfloat16, seed=22, scale=0.05)
    got = torch.full((M, N), float("nan"), dtype=out_dtype, device=DEV)
    splits = tuned().gemm_tiled_splits(M, N, K)
    ws = torch.empty(splits * M * N, dtype=torch.float32, device=DEV) if splits > 1 else None
    tuned().gemm_tiled(x, pack_weight(w), got, ws)
    ref = x.double() @ w.double().T
    scale = ref.abs().max()
    tol = 1e-5 if out_dtype == torch.float32 else 5e-3
    assert (got.double() - ref).abs().max() < tol * scale


@pytest.mark.parametrize("variant", [3, 6, 7, 8, 10, 11, 12, 13, 14, 15, 16, 17])
@pytest.mark.parametrize("M,N,K", [(300, 520, 72), (129, 264, 96), (1100, 640, 256), (400, 452, 1032)])
def test_gemm_tiled_block_shapes(variant, M, N, K):
    """Every block shape of the tiled product (features x tokens: 128 x 96, 128, 160, 224, 256 or 288; 192 x 128 or 224; 224 x 288;
    256 x 160, 224 or 256), whichever the sizes would choose, through the plain epilogue, SwiGLU, the row scale and
    the add-to-the-stream epilogue."""
    from flambeau_amd.kernels.library import load
    from flambeau_amd.kernels.packing import pack_weight
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=23), rnd(N, K, dtype=torch.bfloat16, seed=24, scale=0.05)
    g = 1 + rnd(N, seed=25, scale=0.1)
    resid0 = rnd(M, N, seed=26)
    splits = tuned().gemm_tiled_splits(M, N, K)
    ws = torch.empty(splits * M * N, dtype=torch.float32, device=DEV) if splits > 1 else None
    got = torch.full((M, N), float("nan"), dtype=torch.float32, device=DEV)
    tuned().gemm_tiled(x, pack_weight(w), got, ws, variant=variant)
    ref = x.double() @ w.double().T
    assert (got.double() - ref).abs().max() < 1e-5 * ref.abs().max()
    # a number of K-splits that the sizes would not choose
    ws3 = torch.empty(3 * M * N, dtype=torch.float32, device=DEV)
    got3 = torch.full((M, N), float("nan"), dtype=torch.float32, device=DEV)
    tuned().gemm_tiled(x, pack_weight(w), got3, ws3, variant=variant, splits=3)
    assert (got3.double() - ref).abs().max() < 1e-5 * ref.abs().max()
    # gate and up rows interleaved in fours, activation in the epilogue
    inter = N // 2
    Wgu = tuned().prepare_gate_up(w[:inter].contiguous(), w[inter:2 * inter].contiguous())
    act = torch.full((M, inter), float("nan"), dtype=torch.float32, device=DEV)
    tuned().gemm_tiled(x, Wgu.packed, act, swiglu_rows=Wgu.packed_rows, variant=variant)
    want_act = torch.nn.functional.silu(ref[:, :inter]) * ref[:, inter:2 * inter]
    assert (act.double() - want_act).abs().max() < 2e-5 * want_act.abs().max()
    if splits == 1:
        resid = resid0.clone()
        xg = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
        ssq = torch.full((M, tuned().tiled_parts(M, N, K, variant)), float("nan"), dtype=torch.float32, device=DEV)
        rows = tuned().gemm_tiled_residual(x, pack_weight(w), resid, g, xg, ssq, 1e-5, variant=variant)
        want = resid0.double() + ref
        assert (resid.double() - want).abs().max() < 1e-5 * want.abs().max()
        assert (xg.double() - want * g.double()).abs().max() < 5e-3 * (want * g.double()).abs().max()
        assert (ssq.double().sum(dim=1) - (want * want).sum(dim=1)).abs().max() < 1e-4 * (want * want).sum(dim=1).max()
        # the rows in factors feed a product that scales by the norm itself
        w2 = rnd(200, N, dtype=torch.bfloat16, seed=27, scale=0.05)
        out2 = torch.full((M, 200), float("nan"), dtype=torch.float32, device=DEV)
        sp2 = tuned().gemm_tiled_splits(M, 200, N)
        ws2 = torch.empty(sp2 * M * 200, dtype=torch.float32, device=DEV) if sp2 > 1 else None
        tuned().gemm_tiled(rows.xg, pack_weight(w2), out2, ws2, row_scale=rows, variant=variant)
        normed = want * g.double() * torch.rsqrt((want * want).mean(dim=1, keepdim=True) + 1e-5)
        ref2 = normed @ w2.double().T
        assert (out2.double() - ref2).abs().max() < 1e-2 * ref2.abs().max()


@pytest.mark.parametrize("M,N,K,gate,variant,splits", [(1040, 5120, 32768, False, 11, 2), (384, 16384, 2048, True, 6, 1), (528, 28672, 4096, True, 16, 1),
                                                       (528, 7168, 5120, False, 13, 1), (300, 4096, 14336, False, 13, 4)])
def test_gemm_tiled_plan_knows_what_is_faster(M, N, K, gate, variant, splits):
    """The fastest of all twelve block shapes, whole and in 2 to 6 and 8 parts, at sizes where plans once went a fifth wrong (302 us, 31, 102, 49
    and 52; of 256 x 224, 128 x 224, 224 x 288 and twice 128 x 160; a die that gets one block more than it has units, a block on every unit, which
    lowers the clock): what the plan picks is within a tenth of them.  Weights from memory: enough copies that none stays in a cache."""
    copies = max(2, -(-600_000_000 // (2 * N * K)))
    w = [rnd(N * K, dtype=torch.bfloat16, seed=22, scale=0.05) for _ in range(copies)]       # (N, K multiples of a tile: any values are a packed matrix)
    x, out = rnd(M, K, dtype=torch.bfloat16, seed=21), torch.empty(M, N // 2 if gate else N, dtype=torch.bfloat16, device=DEV)
    ws = torch.empty(8 * M * N, dtype=torch.float32, device=DEV)
    turn = iter(range(1 << 30))
    times = times_in_turn(*(lambda v=v, s=s: tuned().gemm_tiled(x, w[next(turn) % copies], out, ws, swiglu_rows=N if gate else 0, variant=v, splits=s)
                            for v, s in ((variant, splits), (0, 0))))
    assert times[1] < 1.1 * times[0], times


def test_gemm_tiled_splits_k_for_small_grids():
    assert tuned().gemm_tiled_splits(2048, 4096, 4096) == 1
    assert tuned().gemm_tiled_splits(128, 4096, 4096) > 1
    from flambeau_amd.kernels import KernelError
    from flambeau_amd.kernels.packing import pack_weight
    x, w = rnd(128, 4096, dtype=torch.bfloat16), rnd(256, 4096, dtype=torch.bfloat16)
    with pytest.raises(KernelError, match="workspace"):
        tuned().gemm_tiled(x, pack_weight(w), torch.empty(128, 256, dtype=torch.float32, device=DEV))


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("waves", [0, 4, 8])
@pytest.mark.parametrize("M,N,K", [(64, 6144, 4096), (33, 4096, 14336), (17, 250, 96), (48, 37, 2048), (64, 16, 32),
                                   (20, 1000, 160), (1, 300, 64), (49, 16400, 512)])
def test_gemm_mid_against_plain(out_dtype, waves, M, N, K):
    """The kernel for 17 to 64 rows, with both block shapes and with K split or whole."""
    from flambeau_amd.kernels.library import load
    from flambeau_amd.kernels.packing import pack_weight
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=41), rnd(N, K, dtype=torch.bfloat16, seed=42, scale=0.05)
    packed = pack_weight(w)
    ref = x.double() @ w.double().T
    tol = 1e-5 if out_dtype == torch.float32 else 5e-3
    for splits in (0, 1, 3):
        n = tuned().gemm_mid_splits(M, N, K, waves, splits)
        ws = torch.full((n * M * N,), float("nan"), dtype=torch.float32, device=DEV) if n > 1 else None
        got = torch.full((M, N), float("nan"), dtype=out_dtype, device=DEV)
        tuned().gemm_mid(x, packed, got, ws, waves=waves, splits=splits)
        assert (got.double() - ref).abs().max() < tol * ref.abs().max(), (splits, n)


@pytest.mark.parametrize("M,H,I", [(12, 1024, 352), (16, 640, 96), (9, 5120, 64), (40, 544, 48)])
def test_gemm_mid_takes_a_row_scale_in_many_parts(M, H, I):
    """The skinny product leaves a token's sum of squares in a part per 16 features (64 to 320 parts here,
    or 34, which are not read in fours); the kernel for 17 to 64 rows, which large products use from 9 rows on, adds them
    itself before its loop: norm(resid) W^T through the factors equals the formula."""
    from flambeau_amd.kernels.packing import pack_weight
    K0 = 96
    x0, w0 = rnd(M, K0, dtype=torch.bfloat16, seed=31), rnd(H, K0, dtype=torch.bfloat16, seed=32, scale=0.1)
    g = 1 + rnd(H, seed=33, scale=0.1)
    resid = rnd(M, H, seed=34)
    want = resid.double() + x0.double() @ w0.double().T
    xg = torch.full((M, H), float("nan"), dtype=torch.bfloat16, device=DEV)
    if M <= 16:
        ssq = torch.full((M, tuned().skinny_parts(H)), float("nan"), dtype=torch.float32, device=DEV)
        rows = tuned().gemm_skinny_residual(x0, pack_weight(w0), resid, g, xg, ssq, 1e-5)
    else:
        # any producer's parts will do: here 34 parts, which are not read in fours
        r = want.float()
        parts = torch.zeros(M, H // 16, dtype=torch.float32, device=DEV)
        for p_ in range(H // 16):
            parts[:, p_] = (r[:, p_ * 16:(p_ + 1) * 16] ** 2).sum(dim=1)
        resid.copy_(r)
        xg.copy_((r * g).to(torch.bfloat16))
        rows = tuned().NormedRows(xg, parts, 1e-5, resid, g)
    assert rows.ssq.shape[1] > 4
    normed = want * g.double() * torch.rsqrt((want * want).mean(dim=1, keepdim=True) + 1e-5)
    # plain epilogue
    w2 = rnd(200, H, dtype=torch.bfloat16, seed=35, scale=0.05)
    out = torch.full((M, 200), float("nan"), dtype=torch.float32, device=DEV)
    sp = tuned().gemm_mid_splits(M, 200, H)
    ws = torch.empty(sp * M * 200, dtype=torch.float32, device=DEV) if sp > 1 else None
    tuned().gemm_mid(rows.xg, pack_weight(w2), out, ws, row_scale=rows)
    ref = normed @ w2.double().T
    assert (out.double() - ref).abs().max() < 1e-2 * ref.abs().max()
    # gate and up with the activation in the epilogue
    Wgu = tuned().prepare_gate_up(rnd(I, H, dtype=torch.bfloat16, seed=36, scale=0.05), rnd(I, H, dtype=torch.bfloat16, seed=37, scale=0.05))
    act = torch.full((M, I), float("nan"), dtype=torch.bfloat16, device=DEV)
    tuned().gemm_mid(rows.xg, Wgu.packed, act, swiglu_rows=Wgu.packed_rows, row_scale=rows)
    gate = normed @ rnd(I, H, dtype=torch.bfloat16, seed=36, scale=0.05).double().T
    up = normed @ rnd(I, H, dtype=torch.bfloat16, seed=37, scale=0.05).double().T
    want_act = torch.nn.functional.silu(gate) * up
    assert (act.double() - want_act).abs().max() < 2e-2 * want_act.abs().max()


def test_gemm_mid_refuses_what_it_cannot_do():
    from flambeau_amd.kernels import KernelError
    from flambeau_amd.kernels.packing import pack_weight
    out = torch.empty(20, 64, dtype=torch.float32, device=DEV)
    with pytest.raises(KernelError, match="multiple of 32"):
        tuned().gemm_mid(rnd(20, 40, dtype=torch.bfloat16), pack_weight(rnd(64, 40, dtype=torch.bfloat16)), out)
    with pytest.raises(KernelError, match="at most 64"):
        tuned().gemm_mid(rnd(65, 64, dtype=torch.bfloat16), pack_weight(rnd(64, 64, dtype=torch.bfloat16)),
                         torch.empty(65, 64, dtype=torch.float32, device=DEV))
    w = rnd(64, 4096, dtype=torch.bfloat16)
    assert tuned().gemm_mid_splits(20, 64, 4096) > 1
    with pytest.raises(KernelError, match="workspace"):
        tuned().gemm_mid(rnd(20, 4096, dtype=torch.bfloat16), pack_weight(w), out)
    # a K the kernel does not take goes to the skinny kernel through the dispatcher
    w40 = rnd(64, 40, dtype=torch.bfloat16, scale=0.1)
    x40 = rnd(20, 40, dtype=torch.bfloat16)
    tuned().gemm(x40, tuned().prepare_weight(w40), out)
    assert (out.double() - x40.double() @ w40.double().T).abs().max() < 1e-4


@pytest.mark.parametrize("M,nh,nkv,hd,rot,ps,H", [(1, 32, 8, 128, 128, 16, 4096), (8, 4, 2, 16, 16, 8, 64), (16, 5, 5, 32, 16, 16, 80),
                                                  (9, 33, 1, 144, 64, 16, 264),
                                                  (300, 6, 2, 64, 64, 16, 96), (2048, 32, 8, 128, 128, 16, 512),
                                                  (130, 3, 1, 48, 32, 32, 72), (70, 8, 8, 16, 16, 8, 40),
                                                  (64, 32, 8, 128, 128, 16, 4096), (17, 6, 2, 64, 32, 16, 96), (40, 5, 5, 32, 16, 8, 2048),
                                                  (33, 4, 2, 16, 16, 8, 40),
                                                  (512, 32, 8, 128, 128, 16, 4096), (200, 6, 2, 64, 32, 16, 4104), (96, 5, 1, 32, 16, 8, 8192),
                                                  (2600, 32, 8, 128, 128, 16, 4096)])
def test_gemm_with_rotation_and_stores_in_its_kernel(M, nh, nkv, hd, rot, ps, H):
    """The joined q/k/v projection with rows in paired order, rotated and stored by the product's own
    kernel (few rows: skinny; many rows: tiled) or, for 17 to 64 rows and for more rows whose product
    splits K, by a rotation kernel that adds the product's K-splits itself; against product + rotation
    kernel apart and float64."""
    from flambeau_amd.kernels.packing import rotary_paired_rows
    theta = 1e4
    N = (nh + 2 * nkv) * hd
    w = rnd(N, H, dtype=torch.bfloat16, seed=61, scale=0.1)
    x = rnd(M, H, dtype=torch.bfloat16, seed=62)
    order = rotary_paired_rows(nh, nkv, hd, rot).to(DEV)
    W = tuned().prepare_weight(w[order].contiguous())
    # requests of 1 to 40 tokens somewhere in their contexts, pages in a shuffled order
    torch.manual_seed(5)
    pos, seq, starts = [], [], []
    while len(pos) < M:
        k = min(int(torch.randint(1, 41, (1,))), M - len(pos))
        st = int(torch.randint(0, 200, (1,)))
        pos += range(st, st + k); seq += [len(starts)] * k; starts.append(st + k)
    width = max(-(-e // ps) for e in starts) + 1
    n_pages = sum(-(-e // ps) for e in starts) + 2
    perm = torch.randperm(n_pages).int()
    table = torch.full((len(starts), width), -1, dtype=torch.int32)
    used = 0
    for r, e in enumerate(starts):
        nb = -(-e // ps)
        table[r, :nb] = perm[used:used + nb]; used += nb
    pos_d = torch.tensor(pos, dtype=torch.int32, device=DEV)
    seq_d = torch.tensor(seq, dtype=torch.int32, device=DEV)
    table = table.to(DEV)
    angles = torch.empty(M, rot // 2, 2, dtype=torch.float32, device=DEV)
    ops().rope_table(pos_d, rot, theta, angles)
    # apart
    cache_a = make_cache(n_pages, nkv, ps, hd, torch.bfloat16)
    qkv = torch.empty(M, N, dtype=torch.float32, device=DEV)
    tuned().gemm(x, W, qkv)
    q_a = torch.empty(M, nh * hd, dtype=torch.bfloat16, device=DEV)
    ops().rope_kv_write(qkv, pos_d, seq_d, table, q_a, cache_a, nh, rot, theta, table=angles, paired=True)
    # in the product's kernel
    cache_b = make_cache(n_pages, nkv, ps, hd, torch.bfloat16)
    q_b = torch.full((M, nh * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    store = tuned().RopeStore(pos_d, seq_d, table, angles, q_b, cache_b, nh, rot, True)
    if 16 < M <= 64 and H % 32:
        assert not tuned().gemm_rope_store(x, W, store)
        return
    split = M > 64 and tuned().gemm_tiled_splits(M, N, H) > 1
    assert split == ((M, H) in ((512, 4096), (200, 4104), (96, 8192)))          # the cases meant to split do
    assert tuned().gemm_rope_store(x, W, store)
    top = q_a.float().abs().max()
    assert (q_a.float() - q_b.float()).abs().max() <= 2e-2 * top
    assert (cache_a.pool.float() - cache_b.pool.float()).abs().max() <= 2e-2 * cache_a.pool.float().abs().max()
    assert ((cache_a.pool != 0) == (cache_b.pool != 0)).all()          # the same places were written
    if split:
        assert torch.equal(q_a, q_b) and torch.equal(cache_a.pool, cache_b.pool)      # the same sums in the same order
    elif M > 64:
        # every block shape of the tiled product writes the same
        if M == 2600:                                                    # (a size that goes to a block of 288 tokens)
            from flambeau_amd.kernels.library import load
            assert load().fl_gemm_tiled_shape(M, N, H, 1) in (15, 16)
        for variant in (3, 6, 7, 8, 10, 11, 12, 13, 14, 15, 16, 17):
            cache_v = make_cache(n_pages, nkv, ps, hd, torch.bfloat16)
            q_v = torch.full((M, nh * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
            store_v = tuned().RopeStore(pos_d, seq_d, table, angles, q_v, cache_v, nh, rot, True)
            tuned().gemm_tiled_rope(x, W.packed, N, store_v, variant=variant)
            assert torch.equal(q_v, q_b) and torch.equal(cache_v.pool, cache_b.pool), variant
    # float64 reference of q
    ref = (x.double() @ w.double().T)[:, :nh * hd].reshape(M, nh, hd)
    ref = rope_ref(ref, pos_d, theta, rot)
    assert (q_b.double().reshape(M, nh, hd) - ref).abs().max() < 1.5e-2 * ref.abs().max()
    # a layer that reads another layer's cache writes none
    cache_c = make_cache(n_pages, nkv, ps, hd, torch.bfloat16)
    store_c = tuned().RopeStore(pos_d, seq_d, table, angles, torch.empty_like(q_b), cache_c, nh, rot, False)
    assert tuned().gemm_rope_store(x, W, store_c) and not cache_c.pool.any() and torch.equal(store_c.q_out, q_b)


@pytest.mark.parametrize("variant", [3, 7, 16, 17])
def test_gemm_tiled_rotates_into_queries_that_begin_at_8_bytes(variant):
    """Queries and cache pages that begin 8 bytes behind a 16-byte boundary: the bits of those that begin at one, and nothing beside them."""
    from flambeau_amd.kernels.ops import PagedLayerCache
    from flambeau_amd.kernels.packing import pack_weight
    M, nh, nkv, hd, rot, ps, K = 130, 3, 2, 48, 32, 16, 72
    N, pages = (nh + 2 * nkv) * hd, 9
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=62), pack_weight(rnd(N, K, dtype=torch.bfloat16, seed=61, scale=0.1))
    pos, table = torch.arange(M, dtype=torch.int32, device=DEV), torch.arange(pages, dtype=torch.int32, device=DEV)[None].contiguous()
    angles, got = rnd(M, rot // 2, 2, seed=63), []
    for offset in (0, 4):
        room = [torch.full((n + 16,), 7.0, dtype=torch.bfloat16, device=DEV) for n in (M * nh * hd, pages * 2 * nkv * ps * hd)]
        q, pool = (r[offset:r.numel() - 16 + offset] for r in room)
        cache = PagedLayerCache(pool.view(pages, 2, nkv, ps, hd))
        store = tuned().RopeStore(pos, torch.zeros_like(pos), table, angles, q.view(M, nh * hd), cache, nh, rot, True)
        tuned().gemm_tiled_rope(x, w, N, store, variant=variant)
        for r, v in zip(room, (q, pool)):
            assert (r[:offset] == 7.0).all() and (r[v.numel() + offset:] == 7.0).all()
        got.append((q.clone(), pool.clone()))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1]) and (got[0][0] != 7.0).all()


def test_gemm_dispatch_rows_agree_across_kernels():
    """The same rows through the skinny, the middle and the tiled kernel: equal up to float rounding of sums."""
    w = rnd(512, 1024, dtype=torch.bfloat16, seed=23, scale=0.05)
    x = rnd(200, 1024, dtype=torch.bfloat16, seed=24)
    W = tuned().prepare_weight(w)
    big = torch.empty(200, 512, dtype=torch.float32, device=DEV)
    tuned().gemm(x, W, big)
    small = torch.empty(3, 512, dtype=torch.float32, device=DEV)
    tuned().gemm(x[17:20].contiguous(), W, small)
    assert (big[17:20] - small).abs().max() < 1e-5 * big.abs().max()
    middle = torch.empty(40, 512, dtype=torch.float32, device=DEV)       # the kernel for 17 to 64 rows
    tuned().gemm(x[10:50].contiguous(), W, middle)
    assert (big[10:50] - middle).abs().max() < 1e-5 * big.abs().max()


# ---------------------------------------------------------------- tiled attention for portions
def tiles_for(seqs, tile=64):
    rows, at = [], 0
    for s, (_, ql) in enumerate(seqs):
        for off in range(0, ql, tile):
            rows.append((s, at + off, min(tile, ql - off), at + off))         # every row is a row of a tile here
        at += ql
    return torch.tensor(rows, dtype=torch.int32, device=DEV).reshape(-1, 4)


def split_workspace(n_rows, nh, hd, n_split):
    hdp = -(-hd // 32) * 32
    return (torch.full((n_rows * nh * n_split * hdp,), float("nan"), dtype=torch.float32, device=DEV),
            torch.full((n_rows * nh * n_split * 2,), float("nan"), dtype=torch.float32, device=DEV))


@pytest.mark.parametrize("heads_per_wave,n_split", [(0, 1), (1, 1), (0, 3), (2, 7)])
@pytest.mark.parametrize("nh,nkv,hd,ps,window", [(32, 8, 128, 16, 0), (4, 2, 16, 8, 16), (6, 1, 24, 16, 0),
                                                (5, 5, 32, 16, 24), (8, 4, 64, 8, 0), (4, 2, 256, 32, 100),
                                                (6, 3, 40, 64, 37), (2, 1, 160, 128, 0), (8, 2, 96, 16, 70)])
def test_attn_prefill_against_plain_and_reference(nh, nkv, hd, ps, window, heads_per_wave, n_split):
    # (context, queries): a whole prompt, a portion deep in a context, one that starts mid-page,
    # a portion that is no multiple of the tile, a short one
    seqs = [(200, 200), (300, 70), (ps * 5 + 3, 9), (131, 130), (64, 64), (17, 16)]
    case = build_attention_case(torch.bfloat16, nh, nkv, hd, ps, seqs, seed=5)
    n = case["n"]
    scale = 1 / math.sqrt(hd)
    q2 = case["q"].reshape(n, nh * hd)
    out = torch.full((n, nh * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    # with n_split > 1 the keys of every tile are split (some parts are empty: 7 parts of 1 to 5 stages) and merged
    part_o, part_ml = split_workspace(n, nh, hd, n_split) if n_split > 1 else (None, None)
    tuned().attn_prefill(q2, out, case["cache"], tiles_for(seqs), case["pos_d"], case["table"], nh, scale, window,
                         heads_per_wave, n_split=n_split, part_o=part_o, part_ml=part_ml)
    plain = torch.empty_like(out)
    ops().attn_plain(q2, plain, case["cache"], case["pos_d"], case["seq_d"], case["table"], nh, scale, window)
    ref = attention_case_ref(case, scale, window)
    top = ref.abs().max()
    err = (out.double().reshape(n, nh, hd) - ref).abs()
    assert not torch.isnan(out).any()
    assert err.max() < 1e-2 * top, f"worst at {np.unravel_index(int(err.argmax()), err.shape)}"
    assert (out.double() - plain.double()).abs().max() < 1.5e-2 * top


@pytest.mark.parametrize("nh,nkv,hd,ps,window,heads,n_split,softcap,sinks", [
    (32, 8, 128, 16, 0, 0, 1, 0.0, False), (32, 8, 128, 16, 300, 2, 3, 0.0, False), (32, 8, 128, 64, 0, 1, 4, 20.0, True), (6, 1, 24, 16, 0, 1, 2, 0.0, True),
    (8, 2, 64, 8, 0, 4, 1, 0.0, False), (20, 1, 64, 8, 90, 2, 2, 0.0, False), (8, 2, 96, 16, 70, 0, 1, 0.0, False), (5, 5, 32, 16, 24, 1, 5, 0.0, False),
    (4, 2, 256, 32, 100, 2, 2, 9.0, True)])
@pytest.mark.parametrize("rows_of", ["many", "one"])
def test_attn_both_gives_the_bits_of_the_two(nh, nkv, hd, ps, window, heads, n_split, softcap, sinks, rows_of):
    """Tiles and single rows in one launch (numbers of blocks that are no multiples of eight, rows that are split, rows that are not, unused places):
    exactly what the two launches give; heads beyond 128 take those."""
    singles = [(1500, 1), (33, 1), (257, 3), (31, 1)] if rows_of == "many" else [(700, 1)]
    seqs = [(300, 70)] + singles + [(200, 200), (131, 130)]
    case = build_attention_case(torch.bfloat16, nh, nkv, hd, ps, seqs, seed=11)
    n = case["n"]
    q2 = case["q"].reshape(n, nh * hd)
    tiles, single, at = [], [], 0
    for s, (_, ql) in enumerate(seqs):
        if ql > 8:
            tiles += [(s, at + off, min(64, ql - off), at + off) for off in range(0, ql, 64)]
        else:
            single += range(at, at + ql)
        at += ql
    tiles = torch.tensor(tiles, dtype=torch.int32, device=DEV)
    items, firsts = (torch.tensor(a, device=DEV) for a in tuned().balanced_items(decode_rows(case, single).cpu().numpy(), tuned().decode_blocks_per_row(nh, nkv), window))
    sink = torch.linspace(-3, 3, nh, device=DEV) if sinks else None
    args = (nh, 1 / math.sqrt(hd), window)
    extras = dict(softcap=softcap, sink=sink)

    def run(both, merge):
        out = torch.full((n, nh * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
        tile_o, tile_ml = split_workspace(n, nh, hd, n_split) if n_split > 1 else (None, None)
        row_o, row_ml = split_workspace(items.shape[0], nh, hd, 1)
        its, f = (items, firsts) if merge else (torch.cat([decode_rows(case, single)[:, :3], torch.full((len(single), 1), 256, dtype=torch.int32, device=DEV)], 1), None)
        if both:
            tuned().attn_both(q2, out, case["cache"], tiles, case["pos_d"], its, case["table"], *args, heads_per_wave=heads, n_split=n_split, tile_part_o=tile_o,
                              tile_part_ml=tile_ml, row_part_o=row_o, row_part_ml=row_ml, firsts=f, **extras)
        else:
            tuned().attn_prefill(q2, out, case["cache"], tiles, case["pos_d"], case["table"], *args, heads, n_split=n_split, part_o=tile_o, part_ml=tile_ml, **extras)
            tuned().attn_decode(q2, out, case["cache"], its, case["table"], *args, 0, row_o, row_ml, firsts=f, **extras)
        return out

    for merge in (True, False):
        want = run(False, merge)
        assert not torch.isnan(want).any()
        assert torch.equal(run(True, merge), want)


@pytest.mark.parametrize("heads,n_split", [(2, 1), (2, 2), (1, 1)])
def test_attn_both_with_tables_that_leave_a_unit_one_block(heads, n_split):
    """6,000 pages: tiles that fill the chip by themselves, whole (the two launches) or in parts (one)."""
    nh, nkv, hd, ps, window = 32, 8, 128, 16, 0
    seqs = [(1100, 1100), (900, 1), (40, 1)]
    case = build_attention_case(torch.bfloat16, nh, nkv, hd, ps, seqs, seed=12)
    n, q2 = case["n"], case["q"].reshape(case["n"], nh * hd)
    table = torch.full((3, 6000), -1, dtype=torch.int32, device=DEV)
    table[:, :case["table"].shape[1]] = case["table"]
    tiles = torch.tensor([(0, off, min(64, 1100 - off), off) for off in range(0, 1100, 64)], dtype=torch.int32, device=DEV)
    items, firsts = (torch.tensor(a, device=DEV) for a in tuned().balanced_items(decode_rows(case, [1100, 1101]).cpu().numpy(), tuned().decode_blocks_per_row(nh, nkv), window))
    outs = []
    for both, t in ((True, table), (False, table), (True, case["table"])):
        out = torch.full((n, nh * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
        tile_o, tile_ml = split_workspace(n, nh, hd, n_split) if n_split > 1 else (None, None)
        row_o, row_ml = split_workspace(items.shape[0], nh, hd, 1)
        rest = (nh, 1 / math.sqrt(hd), window)
        if both:
            tuned().attn_both(q2, out, case["cache"], tiles, case["pos_d"], items, t, *rest, heads_per_wave=heads, n_split=n_split, tile_part_o=tile_o, tile_part_ml=tile_ml,
                              row_part_o=row_o, row_part_ml=row_ml, firsts=firsts)
        else:
            tuned().attn_prefill(q2, out, case["cache"], tiles, case["pos_d"], t, *rest, heads, n_split=n_split, part_o=tile_o, part_ml=tile_ml)
            tuned().attn_decode(q2, out, case["cache"], items, t, *rest, 0, row_o, row_ml, firsts=firsts)
        outs.append(out)
    assert not torch.isnan(outs[0]).any() and torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


def test_attn_prefill_refuses_page_sizes_it_cannot_take():
    from flambeau_amd.kernels import KernelError
    for ps in (4, 12):
        case = build_attention_case(torch.bfloat16, 2, 1, 16, ps, [(20, 20)], seed=1)
        q2 = case["q"].reshape(20, 32)
        with pytest.raises(KernelError, match="power of two"):
            tuned().attn_prefill(q2, torch.empty_like(q2), case["cache"], tiles_for([(20, 20)]), case["pos_d"],
                                 case["table"], 2, 0.25, 0)
        assert not tuned().prefill_supported(case["cache"], case["table"])     # the engine takes the plain kernel


def test_attn_prefill_peaked_scores_find_single_keys():
    """One key per query is made to stand out (large q.k): the output must be that key's value
    row, wherever the key lies: first key, a page's edge, the window's first key, the query itself."""
    nh, nkv, hd, ps, window = 4, 1, 64, 16, 48
    seqs = [(160, 160)]
    case = build_attention_case(torch.bfloat16, nh, nkv, hd, ps, seqs, seed=6)
    n = 160
    q = torch.zeros(n, nh, hd, dtype=torch.bfloat16, device=DEV)
    targets = []
    K = case["K"][0]
    for i in range(n):
        lo = max(0, i - window + 1)
        t = [lo, i, (i // ps) * ps if (i // ps) * ps >= lo else lo, min(i, lo + 15)][i % 4]
        targets.append(t)
        q[i] = (K[t, 0] / K[t, 0].norm() * 60.0).to(torch.bfloat16)          # all heads alike
    case["q"] = q
    ref = attention_case_ref(case, 1.0, window)
    for n_split in (1, 2):          # whole, and with the keys of every tile in two parts
        out = torch.full((n, nh * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
        part_o, part_ml = split_workspace(n, nh, hd, n_split) if n_split > 1 else (None, None)
        tuned().attn_prefill(q.reshape(n, nh * hd), out, case["cache"], tiles_for(seqs), case["pos_d"], case["table"], nh,
                             1.0, window, n_split=n_split, part_o=part_o, part_ml=part_ml)
        assert (out.double().reshape(n, nh, hd) - ref).abs().max() < 2e-2 * ref.abs().max()
    # and the reference indeed picks single keys
    V = case["V"][0]
    hits = sum(float((ref[i, 0] - V[targets[i], 0]).abs().max()) < 0.05 for i in range(n))
    assert hits > 0.9 * n


def build_long_attention_case(nh, nkv, hd, ps, seqs, width, seed=0):
    """``build_attention_case`` for contexts of tens of thousands of keys (bfloat16): the cache is filled
    with a few indexed copies instead of key by key, the pool starts as NaN (a key read from a page that
    was never written shows), and the block tables are ``width`` wide."""
    g = torch.Generator().manual_seed(seed)
    dtype = torch.bfloat16
    n_pages = sum(-(-c // ps) for c, _ in seqs) + 5
    from flambeau_amd.kernels.ops import PagedLayerCache
    cache = PagedLayerCache(torch.full((n_pages, 2, nkv, ps, hd), float("nan"), dtype=dtype, device=DEV))
    perm = torch.randperm(n_pages, generator=g)
    table = torch.full((len(seqs), width), -1, dtype=torch.int32)
    used, K, V = 0, [], []
    for s, (c, _) in enumerate(seqs):
        nb = -(-c // ps)
        table[s, :nb] = perm[used:used + nb].int()
        used += nb
        k = (torch.randn(c, nkv, hd, generator=g) * 0.8).to(dtype).to(DEV)
        v = torch.randn(c, nkv, hd, generator=g).to(dtype).to(DEV)
        K.append(k.double())
        V.append(v.double())
        t = torch.arange(c, device=DEV)
        page, r = table[s].to(DEV)[t // ps].long(), t % ps
        keys = cache.pool[:, 0].reshape(n_pages, nkv, ps, hd)
        vals = cache.pool[:, 1].reshape(n_pages, nkv, hd, ps)
        keys[page, :, r] = k                      # [c, nkv, hd]
        vals[page, :, :, r] = v                   # values lie transposed inside a page
    pos, tok_seq = [], []
    for s, (c, ql) in enumerate(seqs):
        pos += list(range(c - ql, c))
        tok_seq += [s] * ql
    n = len(pos)
    q = (torch.randn(n, nh, hd, generator=g) * 0.8).to(dtype).to(DEV)
    return dict(cache=cache, table=table.to(DEV), K=K, V=V, pos=pos, tok_seq=tok_seq, q=q, n=n,
                pos_d=torch.tensor(pos, dtype=torch.int32, device=DEV),
                seq_d=torch.tensor(tok_seq, dtype=torch.int32, device=DEV))


@pytest.mark.parametrize("nh,nkv,hd,window", [(4, 2, 64, 0), (2, 1, 128, 0), (4, 2, 64, 5000), (2, 2, 256, 0)])
def test_attn_prefill_with_block_tables_beyond_4096_pages(nh, nkv, hd, window):
    """Portions behind 66,000 to 70,000 keys in pages of 16: block tables 8,192 wide, which a block keeps
    in LDS beside its ring (one block per compute unit then, where two fit with narrower tables).  Random
    queries against the float64 formula and the plain kernel; then queries that each single out one key
    (the first of the context, keys either side of page 4,096, the window's first key, a near one)."""
    ps, width = 16, 8192
    assert tuned().prefill_max_pages(hd) >= width
    seqs = [(70000, 72), (300, 200), (65552, 66)]
    case = build_long_attention_case(nh, nkv, hd, ps, seqs, width, seed=8)
    assert tuned().prefill_supported(case["cache"], case["table"], window)
    n = case["n"]
    scale = 1 / math.sqrt(hd)
    tiles = tiles_for(seqs)
    q2 = case["q"].reshape(n, nh * hd)
    ref = attention_case_ref(case, scale, window)
    top = ref.abs().max()
    plain = torch.empty_like(q2)
    ops().attn_plain(q2, plain, case["cache"], case["pos_d"], case["seq_d"], case["table"], nh, scale, window)
    assert (plain.double().reshape(n, nh, hd) - ref).abs().max() < 1e-2 * top
    for n_split in (1, 5, tuned().attn_prefill_splits(tiles.shape[0], nh, nkv, hd, 70000)):
        out = torch.full((n, nh * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
        part_o, part_ml = split_workspace(n, nh, hd, n_split) if n_split > 1 else (None, None)
        tuned().attn_prefill(q2, out, case["cache"], tiles, case["pos_d"], case["table"], nh, scale, window,
                             n_split=n_split, part_o=part_o, part_ml=part_ml)
        err = (out.double().reshape(n, nh, hd) - ref).abs()
        assert not torch.isnan(out).any(), n_split
        assert err.max() < 1e-2 * top, f"{n_split} splits: worst at {np.unravel_index(int(err.argmax()), err.shape)}"
        assert (out.double() - plain.double()).abs().max() < 1.5e-2 * top
    # peaked: every query of the long requests picks one key, all heads of a kv head alike
    q = case["q"].clone()
    targets = {}
    for i in range(n):
        s, p = case["tok_seq"][i], case["pos"][i]
        if seqs[s][0] < 60000:
            continue
        lo = max(0, p - window + 1) if window else 0
        t = [lo, 65535, 65536, p - 3, lo + 17, 65519][i % 6]
        t = min(max(t, lo), p)
        targets[i] = t
        for h in range(nh):
            k = case["K"][s][t, h // (nh // nkv)]
            q[i, h] = (k / k.norm() * 60.0 / scale / k.norm()).to(torch.bfloat16)       # the score of key t is 60
    case["q"] = q
    ref = attention_case_ref(case, scale, window)
    hits = sum(float((ref[i, 0] - case["V"][case["tok_seq"][i]][t, 0]).abs().max()) < 0.05 for i, t in targets.items())
    assert hits > 0.9 * len(targets)                    # the reference indeed picks single keys
    for n_split in (1, 3):
        out = torch.full((n, nh * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
        part_o, part_ml = split_workspace(n, nh, hd, n_split) if n_split > 1 else (None, None)
        tuned().attn_prefill(q.reshape(n, nh * hd), out, case["cache"], tiles, case["pos_d"], case["table"], nh, scale, window,
                             n_split=n_split, part_o=part_o, part_ml=part_ml)
        assert (out.double().reshape(n, nh, hd) - ref).abs().max() < 2e-2 * ref.abs().max(), n_split


@pytest.mark.parametrize("nh,nkv,hd,window", [(8, 8, 32, 0), (16, 8, 64, 700)])
def test_attn_prefill_grid_that_comes_in_several_rounds(nh, nkv, hd, window):
    """More blocks than the chip holds at once (over 70 tiles of 64 tokens x 8 kv heads): such a grid starts
    the tiles with the most keys first, all head groups of a tile side by side; every (tile, head group)
    must still be taken exactly once.  Three requests, so that the list of tiles is not in order of length."""
    ps = 16
    seqs = [(3000, 3000), (1500, 1300), (200, 150), (77, 77)]
    tiles = tiles_for(seqs)
    assert tiles.shape[0] * nkv > 2 * 256
    case = build_long_attention_case(nh, nkv, hd, ps, seqs, 192, seed=3)
    n = case["n"]
    scale = 1 / math.sqrt(hd)
    q2 = case["q"].reshape(n, nh * hd)
    out = torch.full((n, nh * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    tuned().attn_prefill(q2, out, case["cache"], tiles, case["pos_d"], case["table"], nh, scale, window)
    assert not torch.isnan(out).any()
    plain = torch.empty_like(out)
    ops().attn_plain(q2, plain, case["cache"], case["pos_d"], case["seq_d"], case["table"], nh, scale, window)
    top = plain.double().abs().max()
    assert (out.double() - plain.double()).abs().max() < 1.5e-2 * top
    # the float64 formula at the rows of a few tiles: the longest, one in the middle, the last request's
    rows = list(range(2936, 3000)) + list(range(3000 + 640, 3000 + 704)) + list(range(n - 77, n))
    for i in rows[::3]:
        s_, p_ = case["tok_seq"][i], case["pos"][i]
        ref = attention_ref(case["q"][i].double(), case["K"][s_], case["V"][s_], p_, scale, window)
        assert (out[i].double().reshape(nh, hd) - ref).abs().max() < 1e-2 * top, i


def test_attn_prefill_table_limits_come_from_the_library():
    """Tables wider than a block can keep are refused by the kernel, and the wrapper that chooses the
    kernel asks the same function; with a window only the window's pages count."""
    from flambeau_amd.kernels import KernelError
    t = tuned()
    assert t.prefill_max_pages(128) == 16384 and t.prefill_max_pages(64) == 16384 and 4096 < t.prefill_max_pages(256) < 16384
    case = build_attention_case(torch.bfloat16, 2, 1, 16, 16, [(40, 40)], seed=1)
    wide = torch.full((1, 20000), -1, dtype=torch.int32, device=DEV)
    wide[:, :case["table"].shape[1]] = case["table"]
    assert not t.prefill_supported(case["cache"], wide, 0)
    assert t.prefill_supported(case["cache"], wide, 1000)
    assert t.prefill_supported(case["cache"], wide[:, :16384].contiguous(), 0)
    q2 = case["q"].reshape(40, 32)
    with pytest.raises(KernelError, match="pages per request"):
        t.attn_prefill(q2, torch.empty_like(q2), case["cache"], tiles_for([(40, 40)]), case["pos_d"], wide, 2, 0.25, 0)
    out = torch.full_like(q2, float("nan"))
    t.attn_prefill(q2, out, case["cache"], tiles_for([(40, 40)]), case["pos_d"], wide, 2, 0.25, 24)      # a window: taken
    ref = attention_case_ref(case, 0.25, 24)
    assert (out.double().reshape(40, 2, 16) - ref).abs().max() < 1e-2 * ref.abs().max()


# ---------------------------------------------------------------- gated feed-forward in the product's epilogue
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,I,K", [(1, 14336, 4096), (8, 224, 96), (64, 136, 80), (5, 13, 40), (200, 14336, 512),
                                   (65, 160, 64), (300, 52, 72), (16, 8, 8), (40, 14336, 4096), (23, 100, 96)])
def test_gemm_swiglu_epilogue(out_dtype, M, I, K):
    gate = rnd(I, K, dtype=torch.bfloat16, seed=31, scale=0.3)
    up = rnd(I, K, dtype=torch.bfloat16, seed=32, scale=0.3)
    x = rnd(M, K, dtype=torch.bfloat16, seed=33)
    W = tuned().prepare_gate_up(gate, up)
    assert W.packed is not None and W.swiglu_cols == I and W.packed_rows % 16 == 0
    got = torch.full((M, I), float("nan"), dtype=out_dtype, device=DEV)
    if M <= 64:
        tuned().gemm_skinny(x, W.packed, got, swiglu_rows=W.packed_rows)
    else:
        tuned().gemm_tiled(x, W.packed, got, swiglu_rows=W.packed_rows)
    g, u = x.double() @ gate.double().T, x.double() @ up.double().T
    ref = g / (1 + torch.exp(-g)) * u
    tol = 2e-5 if out_dtype == torch.float32 else 6e-3
    assert (got.double() - ref).abs().max() < tol * ref.abs().max()
    if M <= 64 and K % 32 == 0:
        mid = torch.full((M, I), float("nan"), dtype=out_dtype, device=DEV)
        tuned().gemm_mid(x, W.packed, mid, swiglu_rows=W.packed_rows)
        assert (mid.double() - ref).abs().max() < tol * ref.abs().max()


# ---------------------------------------------------------------- the 32-bit product on the matrix cores
@pytest.mark.parametrize("M,N,K", [(M, N, K) for N, K in [(1, 4), (15, 16), (17, 20), (64, 36), (65, 256), (130, 260), (192, 516), (31, 1040)]
                                   for M in [1, 4, 5, 16, 17, 32, 33, 48, 49, 64, 65, 97, 150]] +
                         [(40, 8192, 100), (40, 8196, 36), (64, 8192, 68), (64, 8260, 516), (33, 4096, 14336)])
def test_gemm_float_gives_the_plain_kernel_s_bits(M, N, K):
    """Every kernel for few rows (to 4, 16, 32 and 48) and for many (16, 32 and 48 a block), both sides of each rule between
    them.  Rows that do not begin at 16 bytes go to the plain kernel, whose sums these are: equal to the last bit."""
    def at(offset, rows, seed):
        buf = torch.empty(rows * K + 4, dtype=torch.float32, device=DEV)
        view = buf[offset:offset + rows * K].view(rows, K)
        view.copy_(rnd(rows, K, seed=seed))
        return view
    want = torch.empty(M, N, dtype=torch.float32, device=DEV)
    ops().gemm_plain(at(1, M, 31), at(0, N, 32), want)
    got = torch.full((M, N), float("nan"), dtype=torch.float32, device=DEV)
    ops().gemm_plain(at(0, M, 31), at(0, N, 32), got)
    assert torch.equal(got, want)


@pytest.mark.parametrize("M,N,K", [(4, 4096, 14336), (16, 4096, 4096), (40, 4096, 1000), (333, 4096, 4096), (100, 4096, 14336), (200, 4096, 100)])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("one_sign", [False, True])
def test_32_bit_products_are_as_close_to_64_bits_as_chains_of_16_with_a_compensated_addition(M, N, K, offset, one_sign):
    """Both kernels on the matrix cores and (rows that do not begin at 16 bytes) the plain one.  The bounds are those chains' own distances,
    2-norm of the difference over 2-norm of the sums: 8.0e-8 at K 100 and 8.1e-8 beyond for normal values; 3.75e-8 at 100, 2.33e-8 at 1000, 2.16e-8 at 4096 and
    2.42e-8 at 14336 where all products have one sign.  The kernels' are 7.5e-8, and the same within 0.3 % with one sign, which half a percent over the bound leaves room for; groups
    of 64 joined in 32 bits are 2 to 18 % beyond the latter at K up to 4096, 32-bit accumulators 2 to 4 times beyond the former.  Single values: seven of these deviations, and the last rounding
    of the largest sums (at most 6 deviations of them, 2^-24 each)."""
    g = torch.Generator(device=DEV).manual_seed(K + M)
    def at(rows, scale):
        view = torch.empty(rows * K + 4, dtype=torch.float32, device=DEV)[offset:offset + rows * K].view(rows, K)
        view.copy_(torch.randn(rows, K, generator=g, device=DEV) * scale)
        return view.abs_() if one_sign else view
    x, w, out = at(M, 1.0), at(N, 0.02), torch.empty(M, N, dtype=torch.float32, device=DEV)
    ops().gemm_plain(x, w, out)
    want = x.double() @ w.double().t()
    off, size = out.double() - want, want.square().mean().sqrt()
    bound = {100: 3.75e-8, 1000: 2.33e-8, 4096: 2.16e-8, 14336: 2.42e-8}[K] * 1.005 if one_sign else 8.0e-8
    assert off.square().mean().sqrt() < bound * size
    assert off.abs().max() < 7 * bound * size + (0.0 if one_sign else 6 * 2 ** -24 * size)


@pytest.mark.parametrize("M,N,K", [(100, 4100, 68), (130, 6148, 100), (47, 28676, 36), (333, 6148, 132), (500, 4100, 20), (16, 28676, 196), (17, 28676, 60)])
def test_gemm_float_blocks_of_one_to_three_tiles_give_the_plain_kernel_s_bits(M, N, K):
    """Sizes at which each number of tiles of x to a block is the cheapest, and where the kernel for few rows ends; K that ends in every kind of chain."""
    test_gemm_float_gives_the_plain_kernel_s_bits(M, N, K)


@pytest.mark.parametrize("M,N,K", [(17, 32768, 32), (32, 16384, 20), (49, 8192, 16), (64, 6144, 32), (40, 8192, 48), (32, 4096, 20)])
def test_gemm_float_takes_short_sums_where_it_is_faster(M, N, K):
    """Measured 0.58 to 0.84 of the plain kernel's time: sizes next to those that it leaves to that one (the test above).  They must not take
    as long as operands that always go there."""
    w, out = rnd(N, K, seed=32), torch.empty(M, N, dtype=torch.float32, device=DEV)
    rows = [torch.empty(M * K + 4, dtype=torch.float32, device=DEV)[offset:offset + M * K].view(M, K).copy_(rnd(M, K, seed=31)) for offset in (0, 1)]
    times = times_in_turn(*(lambda x=x: ops().gemm_plain(x, w, out) for x in rows))
    assert times[0] < 0.93 * times[1], times


@pytest.mark.parametrize("M,N,K", [(8, 256, 16), (1000, 4096, 15)])
def test_gemm_plain_does_no_work_behind_sums_of_up_to_16(M, N, K):
    """Such a sum takes half the products of one of 32 (measured 0.81 and 0.85 of its time, 1.0 with a step of 32 for both)."""
    out = torch.empty(M, N, dtype=torch.float32, device=DEV)
    pairs = [(rnd(M, k, seed=31), rnd(N, k, seed=32)) for k in (K, 2 * K - 1)]       # (rows that do not begin at 16 bytes; 16 k of 8 rows come here as they are)
    times = times_in_turn(*(lambda x=x, w=w: ops().gemm_plain(x, w, out) for x, w in pairs))
    assert times[0] < 0.95 * times[1], times


@pytest.mark.parametrize("M,N,K", [(1, 32768, 32), (8, 16384, 20), (16, 131072, 64), (40, 8192, 16), (64, 6144, 32), (1000, 4096, 16)])
def test_gemm_float_leaves_short_sums_to_the_plain_kernel(M, N, K):
    """Where the blocks' beginnings would take longer than their sums (measured 1.12 to 2.9 times the plain kernel's time):
    no longer than operands that do not begin at 16 bytes, which always go to that one."""
    w, out, times = rnd(N, K, seed=32), torch.empty(M, N, dtype=torch.float32, device=DEV), []
    for offset in (0, 1):
        x = torch.empty(M * K + 4, dtype=torch.float32, device=DEV)[offset:offset + M * K].view(M, K)
        x.copy_(rnd(M, K, seed=31))
        times.append(time_of(lambda: ops().gemm_plain(x, w, out)))
    assert times[0] < 1.08 * times[1] + 0.2, times


# ---------------------------------------------------------------- the tiled product's blocks
@pytest.mark.parametrize("variant", [6, 7, 8, 10, 11, 12, 13, 14, 15, 16, 17])
@pytest.mark.parametrize("M,N,K", [(1, 16, 8), (255, 223, 32), (257, 449, 40), (256, 192, 128), (193, 225, 160), (385, 257, 96), (128, 129, 256), (300, 1000, 104),
                                   (512, 700, 4096)])
def test_gemm_tiled_block_shapes_give_the_same_bits(variant, M, N, K):
    """Every block shape against 128 features x 256 tokens: every output is the same chain over K, so the same bits; one step, fewer and more steps than
    the rings hold, K's and the tiles' remainders."""
    from flambeau_amd.kernels.packing import pack_weight
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=41), rnd(N, K, dtype=torch.bfloat16, seed=42, scale=0.05)
    packed, got = pack_weight(w), []
    for v in (3, variant):
        out = torch.full((M, N), float("nan"), dtype=torch.float32, device=DEV)
        tuned().gemm_tiled(x, packed, out, variant=v, splits=1)
        got.append(out)
    assert torch.equal(*got)


@pytest.mark.parametrize("variant", [3, 6, 7, 8, 10, 11, 12, 13, 14, 15, 16, 17])
@pytest.mark.parametrize("M,N,K,splits", [(97, 130, 8, 1), (300, 100, 40, 1), (129, 264, 96, 1), (225, 48, 104, 1), (289, 257, 192, 1), (100, 16, 64, 1),
                                          (161, 144, 1032, 3), (257, 96, 1056, 4)])
def test_gemm_tiled_where_a_pair_of_steps_is_not_full(variant, M, N, K, splits):
    """x is fetched in pairs of steps of 32: K that ends within a pair, with the next row behind it (NaN: it would show in every
    feature), odd numbers of steps, parts of K of unlike lengths, fewer steps than the rings hold; features and tokens that end within a tile."""
    from flambeau_amd.kernels.packing import pack_weight
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=51), rnd(N, K, dtype=torch.bfloat16, seed=52, scale=0.05)
    bad = torch.arange(M, device=DEV) % 5 == 4
    x[bad] = float("nan")
    out = torch.full((M + 1, N), 7.0, dtype=torch.float32, device=DEV)
    ws = torch.empty(splits * M * N, dtype=torch.float32, device=DEV)
    tuned().gemm_tiled(x, pack_weight(w), out[:M], ws, variant=variant, splits=splits)
    ref = x.double() @ w.double().T
    assert torch.isnan(out[:M][bad]).all() and (out[M] == 7.0).all()
    # (sums of at most 1,056 products in 32 bits: 1e-5 of the largest, as for the tests of the plain sizes)
    assert (out[:M][~bad].double() - ref[~bad]).abs().max() < 1e-5 * ref[~bad].abs().max()


@pytest.mark.parametrize("variant", [3, 6, 7, 8, 10, 11, 12, 13, 14, 15, 16, 17])
@pytest.mark.parametrize("K,splits", [(96, 1), (24, 1), (352, 1), (1056, 3)])
def test_gemm_tiled_fetches_no_weights_behind_the_last_step(variant, K, splits):
    """Odd numbers of steps: the pair's second half multiplies zeros.  What lies there in memory is the next 16 features' first step, made infinite here (and,
    behind the matrix, what is no number): had it been fetched, even x of zero would make NaN of the features before."""
    from flambeau_amd.kernels.packing import pack_weight
    M, N = 70, 400
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=55), rnd(N, K, dtype=torch.bfloat16, seed=56, scale=0.05)
    odd = torch.arange(N, device=DEV) // 16 % 2 == 1
    w[odd, :32] = float("inf")
    packed = pack_weight(w)
    room = torch.full((packed.numel() + (1 << 16),), float("nan"), dtype=torch.bfloat16, device=DEV)
    room[:packed.numel()] = packed.flatten()
    out = torch.empty(M, N, dtype=torch.float32, device=DEV)
    ws = torch.empty(splits * M * N, dtype=torch.float32, device=DEV)
    tuned().gemm_tiled(x, room[:packed.numel()].view(packed.shape), out, ws, variant=variant, splits=splits)
    ref = x.double() @ w[~odd].double().T
    assert not torch.isfinite(out[:, odd]).any()
    assert (out[:, ~odd].double() - ref).abs().max() < 1e-5 * ref.abs().max()              # (sums of at most 1,056 products in 32 bits)


@pytest.mark.parametrize("K", [(1 << 22) - 8, 1 << 22, (1 << 22) + 8, (1 << 23) + 72])
def test_gemm_tiled_takes_rows_of_any_length(K):
    """Rows longer than a block's 32-bit offsets reach, and the longest that they do, through the plain, the stream's and the activation's epilogue.
    Values of -1, 0 and 1: every sum is a whole number below 2^24, so exact in any order.  Rows and features end within a tile; behind both lies what is no number."""
    M, N, steps = 131, 80, -(-K // 32)
    g = torch.Generator(device=DEV).manual_seed(7)
    x = torch.full((M * K + 4096,), float("nan"), dtype=torch.bfloat16, device=DEV)[:M * K].view(M, K)
    for r in range(M):
        x[r] = torch.randint(-1, 2, (K,), generator=g, device=DEV, dtype=torch.int8).bfloat16()
    w = torch.full((N * steps * 32 + 4096,), float("nan"), dtype=torch.bfloat16, device=DEV)[:N * steps * 32]
    tiles = w.view(N // 16, steps, 4, 16, 8)                             # (a tile of 16 features x 32 values of k: lane 16 g + i holds feature i's piece g)
    rows = torch.zeros(N, steps * 32, dtype=torch.bfloat16, device=DEV)
    for r in range(N):
        rows[r, :K] = torch.randint(-1, 2, (K,), generator=g, device=DEV, dtype=torch.int8).bfloat16()
    tiles.copy_(rows.view(N // 16, 16, steps, 4, 8).permute(0, 2, 3, 1, 4))
    ref = torch.zeros(M, N, dtype=torch.float64, device=DEV)
    for at in range(0, K, 1 << 20):
        ref += (x[:, at:at + (1 << 20)].float() @ rows[:, at:min(at + (1 << 20), K)].float().T).double()
    splits = tuned().gemm_tiled_splits(M, N, K)
    ws = torch.empty(max(splits, 3) * M * N, dtype=torch.float32, device=DEV)
    for variant, parts in ((0, 0), (8, 1), (10, 3)):
        out = torch.full((M + 1, N), 7.0, dtype=torch.float32, device=DEV)
        tuned().gemm_tiled(x, w, out[:M], ws, variant=variant, splits=parts)
        assert torch.equal(out[:M].double(), ref) and (out[M] == 7.0).all()
    resid, gain = torch.zeros(M, N, dtype=torch.float32, device=DEV), torch.ones(N, dtype=torch.float32, device=DEV)
    xg, ssq = torch.empty(M, N, dtype=torch.bfloat16, device=DEV), torch.empty(M, tuned().tiled_parts(M, N, K), dtype=torch.float32, device=DEV)
    tuned().gemm_tiled_residual(x, w, resid, gain, xg, ssq, 1e-5, ws)
    assert torch.equal(resid.double(), ref) and torch.equal(xg, ref.bfloat16())
    act = torch.empty(M, N // 2, dtype=torch.float32, device=DEV)
    tuned().gemm_tiled(x, w, act, swiglu_rows=N)
    gate, up = ref.view(M, N // 8, 2, 4).unbind(2)
    want = (gate / (1 + torch.exp(-gate)) * up).reshape(M, N // 2)
    assert ((act.double() - want).abs() <= 4 * 2.0 ** -23 * want.abs() + 1e-30).all()


@pytest.mark.parametrize("M,N,K,cols", [(1286, 16384, 512, 8192), (1175, 16400, 1000, 8195), (2063, 16384, 512, 8180), (842, 28672, 4096, 14336)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gemm_tiled_activation_in_two_launches(dtype, M, N, K, cols):
    """Whole rounds of the first features and the rest in smaller blocks against one launch: the same sums and the same gate, so the same bits, in rows that are
    whole multiples of eight and that are not; nothing behind a row's last column or the last row."""
    from flambeau_amd.kernels.library import load
    lib = load()
    first = lib.fl_gemm_tiled_gate_first(M, N, K)
    assert 0 < first < N and first % 16 == 0 and cols > first // 2
    x = rnd(M, K, dtype=torch.bfloat16, seed=61)
    w = rnd(N * (-(-K // 32) * 32), dtype=torch.bfloat16, seed=62, scale=0.05)           # (any values are a packed matrix)
    if K % 32:
        w.view(N // 16, -1, 64, 8)[:, -1, 16 * (K % 32 // 8):] = 0                      # (the packing's zeros behind K)
    got = []
    for variant in (0, lib.fl_gemm_tiled_shape(M, N, K, 0)):
        out = torch.full((M + 1, cols), 7.0, dtype=dtype, device=DEV)
        tuned().gemm_tiled(x, w, out[:M], swiglu_rows=N, variant=variant)
        assert (out[M] == 7.0).all()
        got.append(out[:M])
    assert torch.equal(*got) and (got[0] != 7.0).any(dim=0).all()


@pytest.mark.parametrize("variant,tokens", [(3, 256), (6, 224), (7, 224), (8, 128), (10, 256), (11, 224), (12, 128), (13, 160), (14, 160), (15, 288), (16, 288), (17, 96)])
def test_gemm_tiled_activation_of_weights_read_once(variant, tokens):
    """A large matrix and one tile of tokens against the same rows beside more (two tiles, whose copies carry no hint): the same bits, for a full tile, one
    row less and a single row, and for a last tile of features that is not full; and against 32 bits."""
    from flambeau_amd.kernels.packing import pack_weight
    N, K = 26640, 4096                                            # (16 * 1665: no block shape's features divide it)
    x = rnd(tokens + 3, K, dtype=torch.bfloat16, seed=71)
    rows = rnd(N, K, dtype=torch.bfloat16, seed=72, scale=0.02)
    w = pack_weight(rows)
    both = torch.empty(tokens + 3, N // 2, dtype=torch.bfloat16, device=DEV)
    tuned().gemm_tiled(x, w, both, swiglu_rows=N, variant=variant)
    for M in (tokens, tokens - 1, 1):
        out = torch.full((M + 1, N // 2), 7.0, dtype=torch.bfloat16, device=DEV)
        tuned().gemm_tiled(x[:M], w, out[:M], swiglu_rows=N, variant=variant)
        assert (out[M] == 7.0).all() and torch.equal(out[:M], both[:M]), M
    z, up = (x.float() @ rows.float().T).view(tokens + 3, N // 8, 2, 4).unbind(2)           # (gate and up in fours)
    ref = (torch.nn.functional.silu(z) * up).reshape(tokens + 3, N // 2)
    assert (both.float() - ref).abs().max() < 2.0 ** -8 * ref.abs().max()          # (a rounding to bf16, sums good to 1e-5)


@pytest.mark.parametrize("gate", ["silu", "gelu_tanh", "gelu", "clamped"])
def test_gemm_tiled_gates_over_the_whole_range(gate):
    """The tiled product's own gates against 64 bits, ups of one.  silu and the clamped gate are quotients of values good to a unit or two of the last place; the two
    gelus are z times a share (of the logistic function, whose argument is rounded, and of the normal distribution) good to 2e-7.  Zeros where e^-z overflows.
    Gates that are infinite or none, as sums that leave 32 bits make them: what the formula gives, as in the kernels for few rows."""
    inf = float("inf")
    z = torch.cat([torch.linspace(-95, 95, 3000), torch.linspace(-6, 6, 3000), torch.linspace(-88.6, -86, 300),
                   torch.tensor([0.0, -0.0, 1e-30, -1e-30, 300.0, -300.0, 3e38, -3e38, inf, -inf, float("nan")])]).to(DEV).bfloat16()
    M = z.numel()
    finite = torch.isfinite(z)
    x = torch.zeros(M, 64, dtype=torch.bfloat16, device=DEV)
    x[:, 0], x[:, 1] = torch.where(finite, z, 0), 1.0
    x[-3:, 2] = torch.tensor([3e38, -3e38, 3e38])                       # (times 128: an infinite sum beside an up of one)
    x[-1, 40] = -3e38
    gate_w, up_w = torch.zeros(8, 64, dtype=torch.bfloat16, device=DEV), torch.zeros(8, 64, dtype=torch.bfloat16, device=DEV)
    gate_w[:, 0], gate_w[:, 2], gate_w[:, 40], up_w[:, 1] = 1.0, 128.0, 128.0, 1.0
    W = tuned().prepare_gate_up(gate_w, up_w)
    def product(x):
        out = torch.empty(x.shape[0], 8, dtype=torch.float32, device=DEV)
        if gate == "clamped":
            assert tuned().gemm_clamped(x, W, out, None, 1.25, inf, 0.5) is not None
        elif x.shape[0] > 64:
            tuned().gemm_tiled(x, W.packed, out, swiglu_rows=W.packed_rows, gate=gate)
        else:
            tuned().gemm_skinny(x, W.packed, out, swiglu_rows=W.packed_rows, gate=gate)
        return out
    got = product(x)
    d = z.double()[:, None].expand(M, 8)
    want = {"silu": lambda v: v / (1 + torch.exp(-v)), "gelu_tanh": lambda v: v / (1 + torch.exp(-2 * 0.7978845608028654 * (v + 0.044715 * v ** 3))),
            "gelu": lambda v: 0.5 * v * torch.special.erfc(-v / 2 ** 0.5), "clamped": lambda v: v / (1 + torch.exp(-1.25 * v)) * 1.5}[gate](d)
    off = (got.double() - want).abs()
    if gate in ("silu", "clamped"):
        # (as far as e^-z stays in 32 bits: silu to -88.7, and the clamped gate, whose exponent is rounded by up to half a unit of 64, to -70)
        ok = finite & (z > (-88.7 if gate == "silu" else -70)) & (z < 2e38)
        assert (off[ok] <= (4 if gate == "silu" else 40) * 2.0 ** -23 * want[ok].abs() + 1e-44).all(), (off[ok] / want[ok].abs()).max()
    else:
        ok = finite & (z > -30)
        assert (off[ok] <= 2e-7 * d[ok].abs() + 1e-44).all(), (off[ok] / d[ok].abs()).max()
    assert (got[finite & (z <= -88)].abs() < 2e-36).all()
    few = product(x[-11:].contiguous())
    assert torch.equal(torch.isnan(got[-11:]), torch.isnan(few)) and torch.equal(torch.isinf(got[-11:]), torch.isinf(few))
    assert (got[-3] == inf).all() and torch.isnan(got[-2]).all() and (gate == "clamped" or torch.isnan(got[-1]).all())         # (min(NaN, limit) is the limit)


@pytest.mark.parametrize("gate", ["silu", "gelu_tanh", "gelu"])
def test_gemm_tiled_gates_are_as_near_to_64_bits_as_the_formulas(gate):
    """The tiled product's own gates in 32 bits against the kernels for few rows, which call the library's functions: over every range the largest
    relative error from 64 bits is no larger.  Any 32-bit gate is a sum of three bfloat16 values; ups of one."""
    G, M, few = 128, 1024, 64
    gate_w, up_w = torch.zeros(G, 3 * G + 32, dtype=torch.bfloat16, device=DEV), torch.zeros(G, 3 * G + 32, dtype=torch.bfloat16, device=DEV)
    i = torch.arange(G, device=DEV)
    gate_w[i, i] = gate_w[i, G + i] = gate_w[i, 2 * G + i] = 1.0
    up_w[:, 3 * G] = 1.0
    W = tuned().prepare_gate_up(gate_w, up_w)
    formula = {"silu": lambda v: v / (1 + torch.exp(-v)), "gelu_tanh": lambda v: v / (1 + torch.exp(-2 * 0.7978845608028654 * (v + 0.044715 * v ** 3))),
               "gelu": lambda v: 0.5 * v * torch.special.erfc(-v / 2 ** 0.5)}[gate]
    for low, high in [(1e-3, 1.4), (1.4, 5.0), (5.0, 80.0), (-0.5, -1e-3), (-1.4, -0.5), (-3.0, -1.4), (-5.0, -3.0)] + ([(-87.0, -5.0), (-88.7, -87.0)] if gate == "silu" else []):
        z = torch.linspace(low, high, M * G, dtype=torch.float64).float().to(DEV).view(M, G)
        x = torch.zeros(M, 3 * G + 32, dtype=torch.bfloat16, device=DEV)
        x[:, :G] = z
        rest = z - x[:, :G].float()
        x[:, G:2 * G] = rest
        x[:, 2 * G:3 * G] = rest - x[:, G:2 * G].float()
        x[:, 3 * G] = 1.0
        assert torch.equal(x[:, :G].double() + x[:, G:2 * G].double() + x[:, 2 * G:3 * G].double(), z.double())
        got, plain = torch.empty(M, G, dtype=torch.float32, device=DEV), torch.empty(M, G, dtype=torch.float32, device=DEV)
        tuned().gemm_tiled(x, W.packed, got, swiglu_rows=W.packed_rows, gate=gate)
        for at in range(0, M, few):
            tuned().gemm_mid(x[at:at + few], W.packed, plain[at:at + few], swiglu_rows=W.packed_rows, gate=gate)
        want = formula(z.double())
        far = [((v.double() - want).abs() / want.abs()).max().item() for v in (got, plain)]
        assert far[0] <= far[1], (low, high, far)


@pytest.mark.parametrize("variant", [3, 7, 11, 12, 14, 15, 17])
@pytest.mark.parametrize("M,inter", [(1, 8), (130, 113), (257, 132), (300, 264), (193, 226)])
def test_gemm_tiled_activation_for_rows_of_any_width(variant, M, inter):
    """Rows of results that are whole multiples of eight, of four and of neither, in tiles of features with four, six,
    seven and eight groups of 16: float results against the formula, bfloat16 results their rounding to the bit."""
    x, w = rnd(M, 72, dtype=torch.bfloat16, seed=43), rnd(2 * inter, 72, dtype=torch.bfloat16, seed=44, scale=0.3)
    W = tuned().prepare_gate_up(w[:inter].contiguous(), w[inter:].contiguous())
    ref = x.double() @ w.double().T
    for gate, f in (("silu", torch.nn.functional.silu), ("gelu_tanh", lambda z: torch.nn.functional.gelu(z, approximate="tanh"))):
        got = []
        for dtype in (torch.float32, torch.bfloat16):
            out = torch.full((M + 1, inter), float("nan"), dtype=dtype, device=DEV)           # (a row behind the last: not written)
            tuned().gemm_tiled(x, W.packed, out[:M], swiglu_rows=W.packed_rows, gate=gate, variant=variant)
            assert torch.isnan(out[M]).all()
            got.append(out[:M])
        want = f(ref[:, :inter]) * ref[:, inter:]
        assert (got[0].double() - want).abs().max() < 2e-5 * want.abs().max()         # (sums of 72 products, the activation at unit slope)
        assert torch.equal(got[0].bfloat16(), got[1])


@pytest.mark.parametrize("variant", [3, 7, 11, 12, 16, 17])
@pytest.mark.parametrize("M,N", [(130, 100), (257, 132), (65, 4), (300, 1028), (193, 226)])
def test_gemm_tiled_stores_rows_of_any_width(variant, M, N):
    """The plain epilogue's bfloat16 rows of a multiple of four values and of neither: the float results' rounding to the bit, nothing behind a row or the last."""
    from flambeau_amd.kernels.packing import pack_weight
    x, w, got = rnd(M, 72, dtype=torch.bfloat16, seed=43), pack_weight(rnd(N, 72, dtype=torch.bfloat16, seed=44, scale=0.3)), []
    for dtype in (torch.float32, torch.bfloat16):
        out = torch.full((M + 1, N), float("nan"), dtype=dtype, device=DEV)
        tuned().gemm_tiled(x, w, out[:M], variant=variant, splits=1)
        assert torch.isnan(out[M]).all()
        got.append(out[:M])
    assert torch.equal(got[0].bfloat16(), got[1])


@pytest.mark.parametrize("gate", [False, True])
def test_gemm_tiled_stores_rows_of_fours_in_fours(gate):
    """bfloat16 rows of 4,100 values beside rows of 4,104, which are stored eight at a time: a third slower at most (value by value they took 1.6 times as long)."""
    M, K, times = 2000, 1024, []
    x = rnd(M, K, dtype=torch.bfloat16, seed=21)
    for N in (4100, 4104):
        rows = -(-(2 * N if gate else N) // 16) * 16
        w, out = rnd(rows * K, dtype=torch.bfloat16, seed=22, scale=0.05), torch.empty(M, N, dtype=torch.bfloat16, device=DEV)       # (any values are a packed matrix)
        times.append(time_of(lambda: tuned().gemm_tiled(x, w, out, swiglu_rows=rows if gate else 0, splits=0 if gate else 1)))
    assert times[0] < 4 / 3 * times[1], times


# ---------------------------------------------------------------- the walk of the linear recurrences
@pytest.mark.parametrize("mode", ["fixed", "delta", "forget", "delta_per_dim", "gated", "written"])
@pytest.mark.parametrize("D,Dv", [(64, 16), (128, 48), (256, 32)])
def test_linear_scan_in_whole_pieces_gives_the_same_bits(mode, D, Dv):
    """Rows that are no whole 16-byte pieces go the general way, one value at a time: equal outputs and states, for
    requests whose tokens end anywhere in a group of four, of 16 and in a run."""
    from types import SimpleNamespace
    H, lens = 2, [1, 3, 4, 7, 16, 18, 31, 32, 33, 70]
    G = 2 if mode == "forget" else 1
    n, S = sum(lens), len(lens)
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    starts, slots = ints([sum(lens[:i]) for i in range(S)]), ints(list(range(S))[::-1])
    step = SimpleNamespace(seq_q_start=starts, seq_q_len=ints(lens), seq_slots=slots)
    v, gates, decay = rnd(n, H * Dv, seed=52), torch.sigmoid(rnd(n, 2 * H, seed=53)), torch.sigmoid(rnd(n, H * D, seed=54) + 2)
    first, got = rnd(S, H * D * Dv, seed=55), []
    for pad in (4, 3):                             # rows a multiple of four floats apart, and not
        q, k = (torch.empty(n, G * D + pad, dtype=torch.float32, device=DEV)[:, :G * D] for _ in range(2))
        q.copy_(rnd(n, G * D, seed=50))
        k.copy_(torch.sigmoid(rnd(n, G * D, seed=51)) if mode == "forget" else torch.nn.functional.normalize(rnd(n, G * D, seed=51), dim=1))
        state, out = first.clone(), torch.full((n, H * Dv), float("nan"), dtype=torch.float32, device=DEV)
        where = (state, starts, step.seq_q_len, slots, out, H, G, D, Dv)
        if mode == "fixed":
            ops().linear_scan(q, k, v, *where, head_decay=torch.tensor([0.97, 0.5], device=DEV))
        elif mode == "delta":
            ops().linear_scan(q, k, v, *where, token_gates=gates)
        elif mode == "forget":
            ops().linear_scan(q, k, v, *where, channel_decay=True)
        elif mode == "delta_per_dim":
            ops().linear_scan(q, k, v, *where, token_gates=gates, key_decay=decay)
        elif mode == "gated":
            ops().linear_scan_gated(q, k, v, decay, state, step, out, H, G, D, Dv, out_scale=0.3)
        else:
            ops().linear_scan_written(q, k, v, gates, torch.tensor([0.7, -1.5], device=DEV), state, step, out, H, G, D, Dv)
        got.append((out, state))
    assert not got[0][0].isnan().any()
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


# ---------------------------------------------------------------- linear recurrences, a chunk of tokens at a time
def _scan_case(mode, H, G, D, Dv, lens, pad=0):
    """Inputs of a recurrence over ragged requests, and ``run(kernels)`` -> (outputs, states)."""
    from types import SimpleNamespace
    n, S = sum(lens), len(lens)
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    step = SimpleNamespace(seq_q_start=ints([sum(lens[:i]) for i in range(S)]), seq_q_len=ints(lens), seq_slots=ints(list(range(S))[::-1]),
                           host=SimpleNamespace(q_lens=lens))
    c = SimpleNamespace(mode=mode, H=H, G=G, D=D, Dv=Dv, lens=lens, step=step)
    rows = torch.empty(n, 2 * G * D + H * Dv + pad, dtype=torch.float32, device=DEV)           # q, k and v as columns of wider rows
    rows.copy_(rnd(n, rows.shape[1], seed=60))
    c.q, c.k, c.v = rows[:, :G * D], rows[:, G * D:2 * G * D], rows[:, 2 * G * D:2 * G * D + H * Dv]
    c.k *= D ** -0.5
    if mode == "delta":                                                                        # (unit keys, as this rule has them)
        c.k.copy_(torch.nn.functional.normalize(c.k.reshape(n, G, D), dim=2).reshape(n, G * D))
    c.head_decay = 1 - 2.0 ** -(3 + torch.arange(H, dtype=torch.float32, device=DEV))
    c.gates = torch.cat([torch.exp(-rnd(n, H, seed=61).abs() * 0.2), torch.sigmoid(rnd(n, H, seed=62))], dim=1).contiguous()
    c.gates[n // 2, 0] = 0.0                                                                   # (a decay may be nothing at all)
    c.key_decay = torch.sigmoid(rnd(n, H * D, seed=63)) ** (1 / 16)
    c.skip, c.state0 = rnd(H, seed=64), rnd(S, H * D * Dv, seed=65)

    def run(kernels):
        state, out = c.state0.clone(), torch.full((n, H * Dv), float("nan"), dtype=torch.float32, device=DEV)
        where = (state, step, out, H, G, D, Dv)
        if mode == "fixed":
            kernels.fixed(c.q, c.k, c.v, c.head_decay, *where)
        elif mode == "delta":
            kernels.delta(c.q, c.k, c.v, c.gates, *where)
        elif mode == "gated":
            kernels.gated(c.q, c.k, c.v, c.key_decay, *where, 0.5)
        else:
            kernels.written(c.q, c.k, c.v, c.gates, c.skip, *where)
        return out, state
    c.run = run
    return c


def _scan_in_64_bits(c):
    H, G, D, Dv = c.H, c.G, c.D, c.Dv
    q, k = (t.double().reshape(-1, G, D).repeat_interleave(H // G, dim=1) for t in (c.q, c.k))
    v, out, states, at = c.v.double().reshape(-1, H, Dv), [], c.state0.double().reshape(-1, H, Dv, D).clone(), 0
    for s, length in enumerate(c.lens):
        S = states[int(c.step.seq_slots[s])]
        for t in range(at, at + length):
            decay = {"fixed": c.head_decay.double()[:, None, None], "gated": c.key_decay[t].double().reshape(H, 1, D),
                     "written": c.gates[t, :H].double()[:, None, None], "delta": c.gates[t, :H].double()[:, None, None]}[c.mode]
            S.mul_(decay)
            u = v[t] - (S * k[t][:, None, :]).sum(-1) if c.mode == "delta" else v[t]
            u = u * c.gates[t, H:].double()[:, None] if c.mode in ("written", "delta") else u
            S.add_(u[:, :, None] * k[t][:, None, :])
            o = (S * q[t][:, None, :]).sum(-1) * (0.5 if c.mode == "gated" else 1.0)
            out.append(o + c.skip.double()[:, None] * v[t] if c.mode == "written" else o)
        at += length
    return torch.stack(out).reshape(at, H * Dv), states.reshape(len(c.lens), -1)


def _scan_sets(max_tokens=4096):
    from types import SimpleNamespace
    from flambeau_amd.kernels import linear_scan as ls
    rt = SimpleNamespace(max_batch_tokens=max_tokens, buffer=lambda name, rows, cols, dtype, max_rows=None: torch.full((rows, cols), float("nan"), dtype=dtype, device=DEV))
    return ls.PlainLinearScan(rt), ls.TunedLinearScan(rt)


@pytest.mark.parametrize("mode", ["fixed", "gated", "written", "delta"])
@pytest.mark.parametrize("H,G,D,Dv,lens", [(2, 2, 64, 16, [256]), (3, 3, 128, 48, [193, 255, 256, 257, 271]), (4, 2, 128, 64, [1, 320, 127, 191, 193, 7, 700]),
                                           (2, 1, 256, 32, [207, 3, 272])])
def test_scan_in_chunks_against_64_bits(mode, H, G, D, Dv, lens):
    """Requests that end anywhere in a chunk and in 16 tokens, beside requests that walk: outputs and states are no further from 64
    bits than the walk's, or than fewer than 40 roundings (a result is a sum of sums, in chains of at most 16 products and trees of
    three, with a factor and a sum behind; a rounding to 24 bits is 2.4e-8 in the root mean square, 40 of them 1.5e-7)."""
    if mode == "gated" and G != H:
        G = H
    c = _scan_case(mode, H, G, D, Dv, lens)
    plain, chunked = _scan_sets()
    want, walk, got = _scan_in_64_bits(c), c.run(plain), c.run(chunked)
    assert not torch.equal(walk[0], got[0])                      # (the chunks did run)
    for w, a, b in zip(want, walk, got):
        err = lambda x: float((x.double() - w).norm() / w.norm())
        assert err(b) < max(err(a), 1.5e-7), (err(a), err(b))
    at = 0
    for length in lens:                                          # (a request that walks: the walk's bits)
        if length < {"gated": 192, "delta": 256}.get(mode, 128):
            assert torch.equal(walk[0][at:at + length], got[0][at:at + length])
        at += length


@pytest.mark.parametrize("mode", ["fixed", "gated", "written", "delta"])
def test_scan_in_chunks_keeps_values_that_are_no_numbers_behind_their_token(mode):
    """A NaN or an infinity in v reaches its own column from its token on, one in k or q nothing before its token."""
    c = _scan_case(mode, 2, 2, 128, 32, [260])
    _, chunked = _scan_sets()
    before, _ = c.run(chunked)
    for t in (0, 5, 15, 16, 70, 127, 199):
        for bad in (float("nan"), float("inf")):
            kept = c.v[t, 3].clone()
            c.v[t, 3] = bad
            out, _ = c.run(chunked)
            c.v[t, 3] = kept
            # (its column's tokens in the same 16 are then summed one by one: 80 sums of 3e-8)
            assert not torch.isfinite(out[t, 3]) and bool(((out[:t, 3] - before[:t, 3]).abs() <= 2.5e-6 * before.abs().max()).all())
            others = [j for j in range(out.shape[1]) if j != 3]
            assert torch.equal(out[:, others], before[:, others])
            for rows in (c.k, c.q):
                kept = rows[t, 7].clone()
                rows[t, 7] = bad
                out, _ = c.run(chunked)
                rows[t, 7] = kept
                # (under the delta rule the whole chunk of such a key is substituted row by row: other sums, as above)
                bound = 2.5e-6 * before.abs().max() if mode == "delta" and rows is c.k else 0.0
                assert bool(((out[:t] - before[:t]).abs() <= bound).all())


@pytest.mark.parametrize("mode", ["fixed", "gated", "written"])
def test_scan_in_chunks_keeps_an_infinite_state(mode):
    """A state that holds an infinity keeps it through whole chunks, as through the walk's tokens: the same outputs and states
    are infinite, none becomes a NaN, and the other columns are those of a finite state."""
    c = _scan_case(mode, 2, 2, 128, 32, [260])
    plain, chunked = _scan_sets()
    before = c.run(chunked)
    for bad in (float("inf"), float("-inf")):
        c.state0.reshape(2, 32, 128)[1, 3, 7] = bad                  # head 1 (head 0 forgets all at one token), column 3
        for w, a, b in zip(c.run(plain), c.run(chunked), before):
            w, a, b = (t.reshape(-1, 2, 32, t.numel() // (t.shape[0] * 64)) for t in (w, a, b))
            assert torch.isinf(w[:, 1, 3]).any() and not torch.isnan(w).any()
            assert torch.equal(torch.isinf(w), torch.isinf(a)) and torch.equal(w[torch.isinf(w)], a[torch.isinf(a)]) and not torch.isnan(a).any()
            others = [j for j in range(32) if j != 3]
            assert torch.equal(a[:, :, others], b[:, :, others])


def test_scan_in_chunks_overflows_at_its_token_and_not_before():
    """The delta rule with three keys so large that what the third corrects is beyond 32 bits, though no product of two keys is:
    tokens before it, in its 16 too, are what the walk makes of them."""
    c = _scan_case("delta", 2, 2, 64, 16, [320])
    plain, chunked = _scan_sets()
    k = c.k.reshape(320, 2, 64)
    k[:, :, 0] = 0
    k /= k.norm(dim=2, keepdim=True)                             # (the others do not see them)
    for t in (3, 9, 21):
        k[t] = 0
        k[t, :, 0] = 1e10
    c.gates[:, :2], c.gates[:, 2:] = 1.0, 1.0
    c.state0.zero_()
    (want, _), (got, _) = c.run(plain), c.run(chunked)
    assert not torch.isfinite(want[21:]).all() and not torch.isfinite(got[21:]).all()
    for t in range(21):                                          # (80 sums of 3e-8, of values as large as the token's largest per head)
        w, a = want[t].reshape(2, 16), got[t].reshape(2, 16)
        assert bool(((w - a).abs() <= 2.5e-6 * w.abs().max(dim=1, keepdim=True).values).all()), t


def test_scan_rows_that_the_chunks_do_not_take_walk():
    """Rows that are no whole 16-byte pieces, and head sizes that the chunked kernels do not know: the walk's bits."""
    plain, chunked = _scan_sets()
    for c in (_scan_case("fixed", 2, 2, 128, 32, [200], pad=3), _scan_case("written", 2, 2, 96, 32, [200]), _scan_case("delta", 2, 2, 128, 32, [260], pad=1), _scan_case("gated", 2, 2, 128, 24, [200])):
        assert all(torch.equal(a, b) for a, b in zip(c.run(plain), c.run(chunked)))


# ---------------------------------------------------------------- the 32-bit attention on the matrix cores
@pytest.mark.parametrize("cap,sinks", [(0.0, False), (3.0, True)])
@pytest.mark.parametrize("nh,nkv,hd,ps,window", [(8, 2, 128, 16, 0), (4, 4, 64, 8, 0), (40, 2, 64, 4, 37), (3, 1, 128, 32, 100), (6, 2, 64, 64, 64)])
def test_attn_float_rows_do_not_depend_on_their_neighbours(nh, nkv, hd, ps, window, cap, sinks):
    """Requests of one token to several blocks of 64 keys, many rows (tiles of several tokens and requests) against each
    row alone, bit for bit, and against the formula in 64 bits; pages in front of the window given back, what lies behind a
    request's last token and in pages of nobody NaN."""
    seqs = [(300, 300), (70, 70), (33, 1), (200, 9), (1, 1), (640, 3), (64, 64), (65, 1), (449, 130)]
    case = build_attention_case(torch.float32, nh, nkv, hd, ps, seqs, seed=4)
    pool, table = case["cache"].pool, case["table"].cpu()
    held = set()
    for s, (c, ql) in enumerate(seqs):
        if window:
            table[s, :max(0, c - ql - window + 1) // ps] = -1
        held |= {int(p) for p in table[s] if p >= 0}
        if c % ps:
            last = int(table[s, c // ps])
            pool[last, 0].reshape(nkv, ps, hd)[:, c % ps:] = float("nan")
            pool[last, 1].reshape(nkv, hd, ps)[:, :, c % ps:] = float("nan")
    for p in set(range(pool.shape[0])) - held:
        pool[p] = float("nan")
    scale, n = 1 / math.sqrt(hd), case["n"]
    sink = rnd(nh, seed=8) if sinks else None
    q, dev_table = case["q"].reshape(n, nh * hd), table.to(DEV)

    def run(rows):
        out = torch.full((len(rows), nh * hd), float("nan"), dtype=torch.float32, device=DEV)
        ops().attn_plain(q[rows].contiguous(), out, case["cache"], case["pos_d"][rows].contiguous(), case["seq_d"][rows].contiguous(),
                         dev_table, nh, scale, window, softcap=cap, sink=sink)
        return out
    everything = run(list(range(n)))
    for i in list(range(0, n, 37)) + [299, 300, n - 1]:
        assert torch.equal(run([i])[0], everything[i]), i
    some = sorted(torch.randperm(n, generator=torch.Generator().manual_seed(1))[:40].tolist())
    assert torch.equal(run(some), everything[some])
    for i in range(0, n, 7):
        s, p = case["tok_seq"][i], case["pos"][i]
        lo = max(0, p - window + 1) if window else 0
        for h in range(nh):
            kv = h // (nh // nkv)
            score = (case["K"][s][lo:p + 1, kv] @ case["q"][i, h].double()) * scale
            score = cap * torch.tanh(score / cap) if cap else score
            if sinks:
                score = torch.cat([score, sink[h:h + 1].double()])
            want = torch.softmax(score, 0)[:p + 1 - lo] @ case["V"][s][lo:p + 1, kv]
            # weights and values sum in float over up to 640 keys: a few roundings of values up to 4
            assert (everything[i, h * hd:(h + 1) * hd].double() - want).abs().max() < 4e-6


def attn_float_case(nh, nkv, hd, ps, seqs, window, edit=None):
    """A 32-bit case after ``edit(case, put_key, put_value)``, its outputs ``[n, nh, hd]`` and the formula's in 64 bits."""
    case = build_attention_case(torch.float32, nh, nkv, hd, ps, seqs, seed=6)
    pool, table = case["cache"].pool, case["table"].cpu()

    def put(kind):
        def into(s, t, kv, d, value):
            page, r = int(table[s, t // ps]), t % ps
            case["KV"[kind]][s][t, kv, d] = value
            (pool[page, 0].reshape(nkv, ps, hd)[kv, r] if kind == 0 else pool[page, 1].reshape(nkv, hd, ps)[kv, :, r])[d] = value
        return into
    if edit:
        edit(case, put(0), put(1))
    n, scale = case["n"], 1 / math.sqrt(hd)
    out = torch.full((n, nh * hd), 7.0, dtype=torch.float32, device=DEV)
    ops().attn_plain(case["q"].reshape(n, nh * hd), out, case["cache"], case["pos_d"], case["seq_d"], case["table"], nh, scale, window)
    return case, out.reshape(n, nh, hd), attention_case_ref(case, scale, window)


@pytest.mark.parametrize("what", ["query", "block", "key", "low block", "low request"])
def test_attn_float_keeps_a_nan(what):
    """A NaN in a query, in all 64 keys of a block or in a row's only key of one: NaN in the rows that see it and nowhere
    else.  Scores of minus infinity weigh nothing; a row that has no other is NaN."""
    seqs = [(200, 200), (65, 65), (130, 1), (300, 2)]

    def edit(case, put_key, put_value):
        case["q"][:, :, 0] = case["q"][:, :, 0].abs() + 0.1
        if what == "query":
            case["q"][77, 3, 40] = float("nan")
        elif what == "key":
            put_key(1, 64, 1, 9, float("nan"))
        for s, keys in {"block": [(0, range(64, 128))], "low block": [(0, range(64, 128)), (3, [256])], "low request": [(1, range(65))]}.get(what, []):
            for t in keys:
                put_key(s, t, 1, 0, float("nan" if what == "block" else "-inf"))
    _, out, ref = attn_float_case(8, 2, 128, 16, seqs, 0, edit)
    assert torch.equal(out.isnan(), ref.isnan()) and ref.isnan().any() == (what != "low block")
    good = ~ref.isnan()
    assert (out.double() - ref)[good].abs().max() < 4e-6         # as for finite inputs: float sums of up to 300 keys


@pytest.mark.parametrize("window", [0, 37])
@pytest.mark.parametrize("nh,nkv,hd,ps", [(16, 4, 128, 16), (6, 6, 64, 8)])
def test_attn_float_values_reach_the_rows_that_see_them(nh, nkv, hd, ps, window):
    """Infinities and NaN among the values, of later tokens of the same tile and in front of a window: the rows
    that see them as the formula has it, every other row to the last bit what it is without them."""
    seqs = [(200, 200), (70, 9), (90, 30)]

    def edit(case, put_key, put_value):
        put_value(0, 70, 1, 5, float("inf"))
        put_value(0, 101, 0, hd - 1, float("nan"))
        put_value(0, 103, 0, hd - 1, float("-inf"))
        put_value(1, 69, 1, 17, float("nan"))
        for d in range(hd):
            put_value(2, 62, 1, d, float("-inf"))
    _, clean, _ = attn_float_case(nh, nkv, hd, ps, seqs, window)
    case, out, ref = attn_float_case(nh, nkv, hd, ps, seqs, window, edit)
    finite = ref.isfinite()
    assert 0 < (~finite).sum() < finite.numel() / 4
    assert torch.equal(out[finite], clean[finite])
    assert torch.equal(out.nan_to_num(7, 8, 9)[~finite], ref.nan_to_num(7, 8, 9).float()[~finite])


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("context", [9, 24, 40, 56, 72, 100, 340])
def test_attn_float_is_as_precise_as_the_plain_kernel(hd, context):
    """Against 64 bits, over 8 requests with contexts around ``context``: no further off than the kernel that takes
    queries which do not begin at 16 bytes (the two errors are known to about 2 %)."""
    nh, nkv, ps, errors = 16, 4, 16, []
    case = build_attention_case(torch.float32, nh, nkv, hd, ps, [(context - i, 2) for i in range(8)], seed=9)
    n, scale = case["n"], 1 / math.sqrt(hd)
    ref = attention_case_ref(case, scale, 0)
    for offset in (0, 1):
        q = torch.empty(n * nh * hd + 4, dtype=torch.float32, device=DEV)[offset:offset + n * nh * hd].view(n, nh * hd)
        q.copy_(case["q"].reshape(n, nh * hd))
        out = torch.empty(n, nh * hd, dtype=torch.float32, device=DEV)
        ops().attn_plain(q, out, case["cache"], case["pos_d"], case["seq_d"], case["table"], nh, scale, 0)
        errors.append(float((out.double().reshape(n, nh, hd) - ref).norm() / ref.norm()))
    assert errors[0] < 1.05 * errors[1], errors


def times_in_turn(*launches, times=20):
    """Microseconds of one launch of each: the second fastest of five runs of a graph of ``times`` launches, the graphs run in turn (a clock that changes
    meanwhile changes for all of them: one behind the other, a product and itself have differed by a tenth)."""
    graphs, runs = [], [[] for _ in launches]
    for launch in launches:
        launch()
        torch.cuda.synchronize()
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1]):
            for _ in range(times):
                launch()
    for _ in range(5):
        for graph, taken in zip(graphs, runs):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            graph.replay()
            end.record()
            end.synchronize()
            taken.append(1000 * begin.elapsed_time(end) / times)
    return [sorted(taken)[1] for taken in runs]


def time_of(launch, times=20):
    return times_in_turn(launch, times=times)[0]


def attn_float_times(nh, nkv, hd, seqs):
    """Times of the matrix-core kernel and of the plain one, which takes queries that do not begin at 16 bytes."""
    case = build_attention_case(torch.float32, nh, nkv, hd, 16, seqs, seed=3)
    n, out = case["n"], torch.empty(case["n"], nh * hd, dtype=torch.float32, device=DEV)
    times = []
    for offset in (0, 1):
        q = torch.empty(n * nh * hd + 4, dtype=torch.float32, device=DEV)[offset:offset + n * nh * hd].view(n, nh * hd)
        q.copy_(case["q"].reshape(n, nh * hd))
        times.append(time_of(lambda: ops().attn_plain(q, out, case["cache"], case["pos_d"], case["seq_d"], case["table"], nh, hd ** -0.5, 0)))
    return times


def test_attn_float_shares_the_keys_of_many_requests_among_its_waves():
    """64 requests of one token with as many key heads as heads: a tile holds tokens of several requests, which its
    waves form together (measured 44 us against 71; one request after the other 229)."""
    fast, plain = attn_float_times(32, 32, 128, [(100, 1)] * 64)
    assert fast < 1.3 * plain, (fast, plain)


@pytest.mark.parametrize("context", [1, 5, 17, 33])
def test_attn_float_takes_no_longer_for_few_keys(context):
    """Eight requests of one token: measured 4 to 6 us, 11 to 13 with every row on the matrix cores (plain 3.7 to 12)."""
    fast, plain = attn_float_times(32, 8, 128, [(context, 1)] * 8)
    assert fast < 1.4 * plain + 1, (fast, plain)


# ---------------------------------------------------------------- kernels that take whole pieces of four values, and any sizes
def _near(got, want, roundings=8):
    """A handful of 32-bit roundings (and, into the eight bits of bfloat16, one of 2^-8) of values of this size."""
    step = 2.0 ** -8 if got.dtype == torch.bfloat16 else 0.0
    assert bool(((got.double() - want).abs() <= roundings * 2.0 ** -23 * want.abs().max() + 1.01 * step * want.abs()).all())


@pytest.mark.parametrize("n", [1, 9, 70])
@pytest.mark.parametrize("H", [4, 1020, 1022, 1024, 2048, 4096, 4100, 8192, 8196])
def test_rows_in_pieces_and_one_by_one(n, H):
    """Scaled embedding rows and the sum of two normed rows: widths that are whole pieces of four or not, of one to eight pieces
    a thread, and beyond."""
    for dtype in (torch.float32, torch.bfloat16):
        table, out = rnd(11, H, dtype=dtype, seed=70), torch.full((n, H), float("nan"), dtype=torch.float32, device=DEV)
        tokens = torch.arange(n, dtype=torch.int32, device=DEV) % 11
        ops().embed_scaled(table, tokens, out, 7.5)
        assert torch.equal(out, table[tokens.long()].float() * 7.5)
    a, b, wa, wb = rnd(n, H, seed=71), rnd(n, H, seed=72, scale=3.0), rnd(H, seed=73), rnd(H, seed=74)
    out = torch.full((n, H), float("nan"), dtype=torch.float32, device=DEV)
    ops().norm_mix(a, wa, 0.7, b, wb, 1.3, out, 1e-5)
    normed = lambda t, w: t.double() * torch.rsqrt((t.double() ** 2).mean(1, keepdim=True) + 1e-5) * w.double()
    _near(out, 0.7 * normed(a, wa) + 1.3 * normed(b, wb))


@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("n,H,D,rot,col", [(3, 2, 128, 128, 0), (70, 3, 64, 24, 4), (5, 1, 128, 20, 0), (2, 2, 30, 30, 0), (9, 16, 128, 64, 3), (4, 2, 128, 0, 8)])
def test_rotate_scale_in_pieces_and_one_by_one(interleaved, n, H, D, rot, col):
    proj = rnd(n, col + 2 * H * D + 5, seed=75)
    angle = rnd(n, max(rot // 2, 1), seed=76).double()
    table = torch.stack([angle.cos(), angle.sin()], dim=-1).float().contiguous()
    outs = [torch.full((n, H * D), float("nan"), dtype=torch.float32, device=DEV) for _ in range(2)]
    ops().rotate_scale(proj, col, col + H * D, table if rot else None, rot, interleaved, 0.5, 2.0, *outs, H, D)
    for out, c, scale in ((outs[0], col, 0.5), (outs[1], col + H * D, 2.0)):
        x = proj[:, c:c + H * D].double().reshape(n, H, D)
        want = x.clone()
        if rot:
            cos, sin = (t.double()[:, None, :] for t in (table[..., 0], table[..., 1]))
            i, k = (slice(0, rot, 2), slice(1, rot, 2)) if interleaved else (slice(0, rot // 2), slice(rot // 2, rot))
            want[..., i], want[..., k] = x[..., i] * cos - x[..., k] * sin, x[..., k] * cos + x[..., i] * sin
        _near(out, (want * scale).reshape(n, H * D))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,H,Dv,ldh,col", [(3, 2, 128, 128, 4), (70, 4, 64, 96, 0), (2, 3, 30, 32, 1), (5, 33, 128, 128, 2), (4, 2, 256, 256, 0)])
def test_gates_of_heads_in_pieces_and_one_by_one(dtype, n, H, Dv, ldh, col):
    x, gate, act = rnd(n, H * ldh, dtype=dtype, seed=77), rnd(n, col + H * Dv + 4, seed=78), {"sigmoid": torch.sigmoid, "silu": torch.nn.functional.silu}
    heads = x.double().reshape(n, H, ldh)[:, :, :Dv]
    for kind in ("sigmoid", "silu"):
        for per_head in (False, True):
            out = torch.full((n, H * Dv), float("nan"), dtype=dtype, device=DEV)
            ops().heads_gate(x, ldh, gate, col, kind, out, H, per_head, 1.25)
            z = gate[:, col:col + (H if per_head else H * Dv)].double().reshape(n, H, -1)
            _near(out, (heads * 1.25 * act[kind](z)).reshape(n, H * Dv))
        y, w = x.float().reshape(n, H, ldh)[:, :, :Dv].contiguous(), rnd(H * Dv, seed=79)
        out = torch.full((n, H * Dv), float("nan"), dtype=dtype, device=DEV)
        ops().headnorm_gate(y.reshape(n, H * Dv), w, gate, col, out, H, 1e-5, gate_kind=kind)
        z = gate[:, col:col + H * Dv].double().reshape(n, H, Dv)
        normed = y.double() * torch.rsqrt((y.double() ** 2).mean(-1, keepdim=True) + 1e-5)
        _near(out, (normed * w.double().reshape(H, Dv) * act[kind](z)).reshape(n, H * Dv))


@pytest.mark.parametrize("lens", [[1024], [300, 1, 2, 5, 700, 8, 9], [3, 4, 1013], [20, 7]])
@pytest.mark.parametrize("G,H,D,Dv", [(4, 12, 128, 128), (4, 16, 64, 32), (2, 16, 128, 48)])
def test_convolution_of_runs_of_tokens(lens, G, H, D, Dv):
    """Steps of many tokens take eight tokens a wave, others one: requests that end anywhere in such a run, one-token requests, kept
    inputs of earlier steps."""
    n, S, C = sum(lens), len(lens), 2 * G * D + H * Dv
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    proj, w, old = rnd(n, C + 2 * H, seed=80), rnd(C, 4, seed=81), rnd(S, 3, C, seed=82)
    a_log, dt_bias, state = rnd(H, seed=83), rnd(H, seed=84), old.reshape(S, 3 * C).clone()
    prep, gates = (torch.full((n, k), float("nan"), dtype=torch.float32, device=DEV) for k in (C, 2 * H))
    starts = [sum(lens[:i]) for i in range(S)]
    seqs = [s for s, length in enumerate(lens) for _ in range(length)]
    ops().conv_prepare(proj, 0, C, C + H, w, a_log, dt_bias, state, 0, ints(seqs), ints(starts), ints(lens), ints(list(range(S))), prep, gates,
                       G, H, D, Dv, 4, 0.3, 1e-6)
    for s, (at, length) in enumerate(zip(starts, lens)):
        x = torch.cat([old[s], proj[at:at + length, :C]]).double()
        y = torch.nn.functional.silu(sum(x[m:m + length] * w[:, m].double() for m in range(4)))
        qk = y[:, :2 * G * D].reshape(length, 2, G, D)
        qk = qk / (qk.square().sum(-1, keepdim=True) + 1e-6).sqrt() * torch.tensor([0.3, 1.0], device=DEV, dtype=torch.float64)[None, :, None, None]
        _near(prep[at:at + length], torch.cat([qk.reshape(length, -1), y[:, 2 * G * D:]], dim=1), 16)
        assert torch.equal(state[s].reshape(3, C), x[-3:].float())
    _near(gates[:, H:], torch.sigmoid(proj[:, C:C + H].double()))
    _near(gates[:, :H], torch.exp(-torch.exp(a_log.double()) * torch.nn.functional.softplus(proj[:, C + H:].double() + dt_bias.double())), 32)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gates_of_heads_one_by_one_take_no_longer(dtype):
    """Few tokens of heads that are no whole pieces of four take a launch's time, as heads that are do: measured 2.6 us both,
    3.3 for the former with as few blocks as the latter needs."""
    times = []
    for Dv in (128, 126):
        x, gate, out = rnd(8, 32 * Dv, dtype=dtype, seed=85), rnd(8, 32 * Dv, seed=86), torch.empty(8, 32 * Dv, dtype=dtype, device=DEV)
        times.append(time_of(lambda: ops().heads_gate(x, Dv, gate, 0, "sigmoid", out, 32), times=50))
    assert times[1] < 1.15 * times[0], times


@pytest.mark.parametrize("n,H", [(2048, 4098), (900, 4098), (300, 1026), (9000, 130)])
def test_embedding_rows_one_by_one_on_both_sides(n, H):
    """Rows that are no whole pieces of four, over several blocks while the chip holds them all and a block each beyond: every
    value is written."""
    tokens = torch.arange(n, dtype=torch.int32, device=DEV) % 64
    for dtype in (torch.float32, torch.bfloat16):
        table, out = rnd(64, H, dtype=dtype, seed=87), torch.full((n, H), float("nan"), dtype=torch.float32, device=DEV)
        ops().embed_scaled(table, tokens, out, 2.0)
        assert torch.equal(out, table[tokens.long()].float() * 2.0)


def test_convolution_takes_no_leap_where_runs_begin():
    """A few tokens more take no longer than a few tokens more: 8 + 8 + 16 heads of 64, measured 11.0 us for 504 and for 512 tokens,
    14.0 for 512 when they went in runs of eight with half of every wave's loads for nothing."""
    G, H, D, times = 8, 16, 64, []
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    for n in (504, 512):
        C = 2 * G * D + H * D
        proj, w, state = rnd(n, C + 2 * H, seed=88), rnd(C, 4, seed=89), rnd(1, 3 * C, seed=90)
        a_log, dt_bias = rnd(H, seed=91), rnd(H, seed=92)
        prep, gates = (torch.empty(n, k, dtype=torch.float32, device=DEV) for k in (C, 2 * H))
        meta = (ints([0] * n), ints([0]), ints([n]), ints([0]))
        times.append(time_of(lambda: ops().conv_prepare(proj, 0, C, C + H, w, a_log, dt_bias, state, 0, *meta, prep, gates, G, H, D, D, 4, 0.3, 1e-6)))
    assert times[1] < 1.15 * times[0], times


# ---------------------------------------------------------------- between a projection and attention, many tokens
@pytest.mark.parametrize("D,nh,nkv,ps,n,rot,interleaved,head_norm,mix,whole_norm,bias", [
    (128, 32, 8, 16, 200, 128, False, 0, 0, False, False), (128, 5, 3, 16, 745, 64, False, 1, 1, False, True), (64, 6, 2, 8, 1650, 64, True, 2, 2, False, False),
    (256, 3, 1, 32, 820, 128, True, 1, 2, False, True), (64, 7, 5, 64, 965, 16, False, 0, 1, True, False), (128, 4, 0, 16, 2049, 128, False, 2, 0, False, False),
    (256, 2, 2, 24, 691, 0, False, 2, 2, False, False), (128, 8, 2, 8, 700, 8, True, 0, 0, True, True), (128, 5, 3, 16, 744, 64, False, 1, 1, False, True),
    (64, 6, 2, 8, 130, 64, True, 2, 2, False, False)])
def test_qkv_prepare_of_many_tokens(D, nh, nkv, ps, n, rot, interleaved, head_norm, mix, whole_norm, bias):
    """Steps of 2^20 values and more (the last two: just fewer, and far fewer) against the same tokens at most 64 at a time (a wave per head): queries, cache pages and kept values. Requests that begin
    anywhere in a page, some rows without a page; columns behind others. The sums of squares are in another order and the rotations' products may be fused
    otherwise: one rounding to bfloat16 at most, and one unit of 32 bits of what cancels."""
    ops_ = ops()
    torch.manual_seed(n)
    has_kv = nkv > 0
    kv = max(nkv, 1)
    ld = 8 + nh * D + 2 * kv * D
    cols = (8, 8 + nh * D if has_kv else -1, 8 + (nh + kv) * D if has_kv else -1)
    proj = torch.randn(n, ld, device=DEV)
    pos, seq, r = [], [], 0
    while len(pos) < n:                                   # requests of up to 90 tokens, begun anywhere
        k, st = min(int(torch.randint(1, 91, (1,))), n - len(pos)), int(torch.randint(0, 50, (1,)))
        pos += range(st, st + k); seq += [r] * k; r += 1
    width = (50 + 91) // ps + 1
    perm = torch.randperm(r * width).reshape(r, width).int()
    if r > 1: perm[r // 2] = -1                           # (padding rows have no page)
    pos, seq, table = torch.tensor(pos, dtype=torch.int32, device=DEV), torch.tensor(seq, dtype=torch.int32, device=DEV), perm.to(DEV)
    angle = torch.rand(n, max(rot // 2, 1), device=DEV) * 6.3
    cs = torch.stack([angle.cos(), angle.sin()], -1)[:, :rot // 2].contiguous()
    gain = lambda m: 1 + 0.1 * torch.randn(m, device=DEV)
    gq, gk = (gain(nh * D), gain(kv * D) if has_kv else None) if whole_norm else (None, None)
    hq, hk = (gain(D), gain(D)) if head_norm and D != 64 else (None, None)
    b = torch.randn(ld, device=DEV) if bias else None
    kept, lam = torch.randn(n, kv * D, device=DEV), torch.tensor([0.3], device=DEV)
    def run(step):
        cache = make_cache(r * width + 1, kv, ps, D, torch.bfloat16)
        q, first = torch.full((n, nh * D), float("nan"), dtype=torch.bfloat16, device=DEV), kept.clone()
        for at in range(0, n, step):
            s = slice(at, min(at + step, n))
            m = s.stop - at
            q_s, f_s = torch.empty(m, nh * D, dtype=torch.bfloat16, device=DEV), first[s].clone()
            ops_.qkv_prepare(proj[s].contiguous(), cols, pos[s].contiguous(), seq[s].contiguous(), table, q_s, cache, nh, D, D, rot, interleaved,
                             cs[s].contiguous() if rot else None, gq, gk, head_norm, 1e-5, v_first=f_s if mix else None, value_mix=mix, mix=lam if mix == 2 else None,
                             write_cache=has_kv, row_scales=torch.empty(m, 2, device=DEV), q_head_gain=hq, k_head_gain=hk, bias=b)
            q[s], first[s] = q_s, f_s
        return q.float(), cache.pool.float(), first
    (q1, c1, f1), (q2, c2, f2) = run(n), run(64)
    assert torch.equal(f1, f2) and torch.equal(c1 != 0, c2 != 0)
    for a, w in ((q1, q2), (c1, c2)):
        assert ((a - w).abs() <= 2.0 ** -7 * w.abs() + 2.0 ** -20 * w.abs().max()).all()          # (neighbours of 8 significant bits lie at most 2^-7 apart)
    if has_kv:                                            # (values are neither normed nor turned: the same bits)
        assert torch.equal(c1[:, 1], c2[:, 1]) and (c1 != 0).any()


@pytest.mark.parametrize("nh,nkv,D", [(2, 1, 128), (8, 2, 64), (8, 1, 128)])
def test_qkv_prepare_takes_no_leap_behind_64_tokens(nh, nkv, D):
    """A decode step of 65 requests beside one of 64, which a wave per head does: no leap (where the kernel for many tokens began there it took a third longer)."""
    times = []
    for n in (64, 65):
        proj, angles = rnd(n, (nh + 2 * nkv) * D, seed=5), rnd(n, D // 2, 2, seed=6)
        seq, pos = torch.arange(n, dtype=torch.int32, device=DEV), torch.full((n,), 5, dtype=torch.int32, device=DEV)
        cache, q = make_cache(n, nkv, 16, D, torch.bfloat16), torch.empty(n, nh * D, dtype=torch.bfloat16, device=DEV)
        table = seq[:, None].contiguous()
        times.append(time_of(lambda: ops().qkv_prepare(proj, (0, nh * D, (nh + nkv) * D), pos, seq, table, q, cache, nh, D, D, D, False, angles, None, None, 0, 1e-5)))
    assert times[1] < 1.12 * times[0] + 0.1, times
