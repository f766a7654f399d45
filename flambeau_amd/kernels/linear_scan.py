"""The kernel set of the linear recurrences: S <- g S + k u^T, o = S^T q per head, u = v, a part of v, or the delta rule's.

``PlainLinearScan`` walks token by token (``fl_linear_scan*``), which gives a prompt cut anywhere the same bits.
``TunedLinearScan`` takes requests of many tokens 64 at a time on the 32-bit matrix cores (``fl_linear_scan_chunked``): the same
sums in another order, in 32 bits, nearer to 64 bits than the walk's.  Requests of few tokens, steps whose walk is the faster way
(``chunked_from``), and sizes, strides or addresses that the chunked kernels do not take, walk."""
from __future__ import annotations

from typing import NamedTuple

import torch

from . import ops
from .library import call, load
from .sets import register_kernel_set


class PlainLinearScan:
    def __init__(self, rt):
        self.rt = rt

    def fixed(self, q, k, v, head_decay, state, step, out, n_heads, n_qk_heads, dim, vdim):
        """A decay per head, u = v (``ops.linear_scan``)."""
        return ops.linear_scan(q, k, v, state, step.seq_q_start, step.seq_q_len, step.seq_slots, out, n_heads, n_qk_heads, dim, vdim,
                               head_decay=head_decay)

    def delta(self, q, k, v, gates, state, step, out, n_heads, n_qk_heads, dim, vdim):
        """The delta rule with a decay and a write strength per token and head (``ops.linear_scan``)."""
        return ops.linear_scan(q, k, v, state, step.seq_q_start, step.seq_q_len, step.seq_slots, out, n_heads, n_qk_heads, dim, vdim,
                               token_gates=gates)

    def gated(self, q, k, v, key_decay, state, step, out, n_heads, n_qk_heads, dim, vdim, out_scale: float = 1.0):
        """A decay per token, head and key dim (``ops.linear_scan_gated``)."""
        return ops.linear_scan_gated(q, k, v, key_decay, state, step, out, n_heads, n_qk_heads, dim, vdim, out_scale)

    def written(self, q, k, v, gates, skip, state, step, out, n_heads, n_qk_heads, dim, vdim):
        """A decay and a write strength per token and head (``ops.linear_scan_written``)."""
        return ops.linear_scan_written(q, k, v, gates, skip, state, step, out, n_heads, n_qk_heads, dim, vdim)


class Form(NamedTuple):
    """Where the chunks of a form take less time than its walk (``chunked_from``)."""
    tokens: int                    # least tokens of a request
    fill: float                    # few blocks: least share of its chunks that the longest request fills
    ratio: float                   # a full chip: a token's time in whole chunks over its time walked, ratio + per_head * 16 / vdim,
    per_head: float                # (what is prepared per head is shared by the blocks of its vdim / 16 columns)
    half: float                    # times this with two to four blocks per unit,
    wide: float                    # times this with 256 key dims


# Measured one by one over 64, 128 and 256 key dims, 64 and 128 values, 4 to 64 heads, 1 to 64 requests of 96 to 2,048 tokens, 4,800 in
# all.  One request of 16 to 32 heads of 128, us walked and in chunks: a decay per head at 96, 129, 192, 384 tokens 18.8, 23.8, 34.2,
# 62.8 and 20.2, 22.2, 22.7, 31.2; with write strengths 19.0, 24.4, 32.5, 62.8 and 19.8, 22.3, 23.0, 32.2; a decay per key dim, whose
# chunks are more work to prepare, 24.3, 30.7, 39.4, 68.4 and 29.2, 33.3, 34.6, 45.9; the delta rule at 129, 192, 256, 2,048 tokens 37.9,
# 48.0, 61.2, 380 and 52.0, 52.3, 58.8, 199.  A walk's time is its chain's while units are left, so that requests beside it cost nothing;
# with blocks on all of them (512: two a unit) both go by the work there is, and the walk does no more for tokens that do not fill a
# chunk: 64 requests of 129 tokens, 32 heads of 128 x 64, a decay per head 362 and 454, 16 requests of 257 tokens, 64 heads of 64 x 64, the
# delta rule 272 and 493.  Of the 4,800 these rules leave 25 more than 3 % slower than the walk, the worst 12 %; by the least tokens
# alone 494 were, by up to 82 %.
FORMS = {"fixed": Form(128, 0.0, 0.49, 1.62, 0.82, 0.85), "written": Form(128, 0.0, 0.56, 0.9, 0.89, 0.7),
         "gated": Form(192, 0.8, 0.7, 1.27, 0.83, 0.91), "delta": Form(256, 0.84, 0.94, 0.67, 0.93, 1.0)}
FULL_CHIP = 512


def chunks(q_lens, enough: int, size: int) -> int:
    """How many chunks of ``size`` tokens the requests of at least ``enough`` go in: a record each."""
    return sum(-(-q // size) for q in q_lens if q >= enough)


def most_chunks(tokens: int, enough: int, size: int) -> int:
    """The most that ``chunks`` can be for a step of ``tokens``: a chunk per ``size`` of them, and one that is not full per request."""
    return tokens // size + tokens // enough


def chunked_from(kind: str, q_lens, n_heads: int, dim: int, vdim: int, size: int) -> int:
    """From how many tokens on the requests of a step go in chunks of ``size``; 0: all of them walk."""
    form, longest = FORMS[kind], max(q_lens)
    if longest < form.tokens:
        return 0
    count, most = chunks(q_lens, form.tokens, size), -(-longest // size)
    blocks = n_heads * vdim / 16 * count / most                        # at a time, over the longest request's chunks
    if kind == "delta" and blocks >= 2 * dim and longest < form.tokens + size:
        return 0                                                       # (the chunks' preparation beside a short walk: 256 tokens of 64 heads of 64 x 128 48.7 us walked, 58.1)
    if blocks < FULL_CHIP:
        return form.tokens if longest >= form.fill * size * most else 0
    ratio = (form.ratio + form.per_head * 16 / vdim) * (form.half if blocks < 2 * FULL_CHIP else 1.0) * (form.wide if dim == 256 else 1.0)
    return form.tokens if sum(q for q in q_lens if q >= form.tokens) >= ratio * size * count else 0


class TunedLinearScan(PlainLinearScan):
    def _chunked(self, q, k, v, state, step, out, H, G, D, Dv, head_decay=None, gates=None, skip=None, key_decay=None, out_scale=1.0,
                 corrects=False):
        """Whether the chunked kernels did it."""
        kind = "delta" if corrects else "gated" if key_decay is not None else "written" if gates is not None else "fixed"
        lib = load()
        size = lib.fl_linear_scan_chunk_tokens()
        rows = [q, k] + ([key_decay] if key_decay is not None else [])
        enough = chunked_from(kind, step.host.q_lens, H, D, Dv, size)
        if not enough or not lib.fl_linear_scan_chunked_takes(int(D), int(Dv)):
            return False
        if any(t.data_ptr() % 16 or t.stride(0) % 4 for t in rows + [state]) or max(t.stride(0) for t in rows + [v]) >= 1 << 22:
            return False
        n, S = out.shape[0], step.seq_q_start.shape[0]
        f = lambda t, name, shape: ops._check(t, "linear_scan." + name, torch.float32, shape)
        i = lambda t, name: ops._check(t, "linear_scan." + name, torch.int32, (S,))
        count = chunks(step.host.q_lens, enough, size)
        records = self.rt.buffer("scan_records", count, lib.fl_linear_scan_record_floats(int(H), int(D), 1 if key_decay is not None else 2 if corrects else 0),
                                 torch.float32, max_rows=most_chunks(self.rt.max_batch_tokens, enough, size))
        pg = f(gates, "gates", (n, 2 * H)) if gates is not None else None
        call("fl_linear_scan_chunked", *ops._rows(q, "linear_scan.q", n, G * D), *ops._rows(k, "linear_scan.k", n, G * D),
             *ops._rows(v, "linear_scan.v", n, H * Dv), f(head_decay, "decay", (H,)) if head_decay is not None else None,
             pg, pg + 4 * H if pg is not None else None, 2 * H if pg is not None else 0, int(corrects),
             *(ops._rows(key_decay, "linear_scan.key_decay", n, H * D) if key_decay is not None else (None, 0)), float(out_scale),
             f(skip, "skip", (H,)) if skip is not None else None, f(state, "state", (None, None)), state.shape[1],
             i(step.seq_q_start, "seq_q_start"), i(step.seq_q_len, "seq_q_len"), i(step.seq_slots, "seq_slots"), f(out, "out", (n, H * Dv)),
             records.data_ptr(), count, S, enough, int(min(step.host.q_lens) < enough), int(H), int(G), int(D), int(Dv), ops.stream_handle())
        return True

    def fixed(self, q, k, v, head_decay, state, step, out, n_heads, n_qk_heads, dim, vdim):
        where = (q, k, v, state, step, out, n_heads, n_qk_heads, dim, vdim)
        if self._chunked(*where, head_decay=head_decay):
            return out
        return super().fixed(q, k, v, head_decay, state, step, out, n_heads, n_qk_heads, dim, vdim)

    def gated(self, q, k, v, key_decay, state, step, out, n_heads, n_qk_heads, dim, vdim, out_scale: float = 1.0):
        if self._chunked(q, k, v, state, step, out, n_heads, n_qk_heads, dim, vdim, key_decay=key_decay, out_scale=out_scale):
            return out
        return super().gated(q, k, v, key_decay, state, step, out, n_heads, n_qk_heads, dim, vdim, out_scale)

    def delta(self, q, k, v, gates, state, step, out, n_heads, n_qk_heads, dim, vdim):
        if self._chunked(q, k, v, state, step, out, n_heads, n_qk_heads, dim, vdim, gates=gates, corrects=True):
            return out
        return super().delta(q, k, v, gates, state, step, out, n_heads, n_qk_heads, dim, vdim)

    def written(self, q, k, v, gates, skip, state, step, out, n_heads, n_qk_heads, dim, vdim):
        if self._chunked(q, k, v, state, step, out, n_heads, n_qk_heads, dim, vdim, gates=gates, skip=skip):
            return out
        return super().written(q, k, v, gates, skip, state, step, out, n_heads, n_qk_heads, dim, vdim)


register_kernel_set("linear_scan", PlainLinearScan, TunedLinearScan)
