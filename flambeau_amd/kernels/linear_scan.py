"""The kernel set of the linear recurrences: S <- g S + k u^T, o = S^T q per head, u = v, a part of v, or the delta rule's.

``PlainLinearScan`` walks token by token (``fl_linear_scan*``), which gives a prompt cut anywhere the same bits.
``TunedLinearScan`` takes requests of many tokens 64 at a time on the 32-bit matrix cores (``fl_linear_scan_chunked``): the same
sums in another order, in 32 bits, nearer to 64 bits than the walk's.  Requests of few tokens, and sizes, strides or addresses that
the chunked kernels do not take, walk."""
from __future__ import annotations

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


# From this many tokens of a request on its chunks take less time than its walk (us for 96, 129, 192, 384 tokens, 16 to 32 heads: a
# decay per head 18.8, 23.8, 34.2, 62.8 walked and 20.2, 22.2, 22.7, 31.2 in chunks; with write strengths 19.0, 24.4, 32.5, 62.8 and
# 19.8, 22.3, 23.0, 32.2; a decay per key dim, whose chunks are more work to prepare, 24.3, 30.7, 39.4, 68.4 and 29.2, 33.3, 34.6, 45.9;
# the delta rule at 129, 192, 256, 2,048 tokens 37.9, 48.0, 61.2, 380 and 52.0, 52.3, 58.8, 199).
CHUNKED_TOKENS = 128
CHUNKED_TOKENS_PER_DIM = 192
CHUNKED_TOKENS_DELTA = 256


def lengths(batch, enough: int):
    """``(whether a request has enough tokens for chunks, whether one has not)``."""
    return max(batch.q_lens) >= enough, min(batch.q_lens) < enough


def chunks(q_lens, enough: int, size: int) -> int:
    """How many chunks of ``size`` tokens the requests of at least ``enough`` go in: a record each."""
    return sum(-(-q // size) for q in q_lens if q >= enough)


def most_chunks(tokens: int, enough: int, size: int) -> int:
    """The most that ``chunks`` can be for a step of ``tokens``: a chunk per ``size`` of them, and one that is not full per request."""
    return tokens // size + tokens // enough


class TunedLinearScan(PlainLinearScan):
    def _chunked(self, q, k, v, state, step, out, H, G, D, Dv, head_decay=None, gates=None, skip=None, key_decay=None, out_scale=1.0,
                 corrects=False):
        """Whether the chunked kernels did it."""
        enough = CHUNKED_TOKENS_DELTA if corrects else CHUNKED_TOKENS if key_decay is None else CHUNKED_TOKENS_PER_DIM
        long, short = lengths(step.host, enough)
        lib = load()
        rows = [q, k] + ([key_decay] if key_decay is not None else [])
        if not long or not lib.fl_linear_scan_chunked_takes(int(D), int(Dv)):
            return False
        if any(t.data_ptr() % 16 or t.stride(0) % 4 for t in rows + [state]) or max(t.stride(0) for t in rows + [v]) >= 1 << 22:
            return False
        n, S = out.shape[0], step.seq_q_start.shape[0]
        f = lambda t, name, shape: ops._check(t, "linear_scan." + name, torch.float32, shape)
        i = lambda t, name: ops._check(t, "linear_scan." + name, torch.int32, (S,))
        size = lib.fl_linear_scan_chunk_tokens()
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
             records.data_ptr(), count, S, enough, int(short), int(H), int(G), int(D), int(Dv), ops.stream_handle())
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
