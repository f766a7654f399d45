"""The lists that give every single row of a batch splits of its own for the decode attention
(host side only): every row present with consecutive splits, the budget kept, no split shorter than
the least, the list's length a function of the batch's shape alone."""
import random

import numpy as np

from flambeau_amd.kernels import tuned


def test_every_row_gets_consecutive_splits_within_the_budget():
    rng = np.random.default_rng(0)
    for _ in range(1500):
        n = int(rng.integers(1, 70))
        per_row = int(rng.choice([1, 2, 8, 16, 64]))
        pos = rng.integers(0, int(rng.choice([50, 300, 5000, 70000])), n)
        window = int(rng.choice([0, 0, 64, 4096]))
        rows = np.stack([np.arange(n), pos, np.arange(n), np.zeros(n, int)], 1).astype(np.int32)
        items, firsts = tuned.balanced_items(rows, per_row, window)
        assert len(items) == tuned.decode_item_budget(n, per_row)
        used = items[items[:, 0] >= 0]
        assert (items[len(used):, 0] < 0).all()                       # the unused places are the last ones
        by_row = {}
        for r, p, q, w in used:
            assert p == pos[r] and q == r
            by_row.setdefault(int(r), []).append(int(w))
        assert list(by_row) == list(range(n))                          # in the order of the rows
        for r, ws in by_row.items():
            k = ws[0] >> 8
            assert [w & 255 for w in ws] == list(range(k)) and all(w >> 8 == k for w in ws)
            keys = min(pos[r] + 1, window) if window else pos[r] + 1
            assert 1 <= k <= tuned.DECODE_MAX_SPLITS and (k == 1 or keys / k > tuned.DECODE_MIN_KEYS_PER_SPLIT / 2)
        assert all(items[f, 0] == r and items[f, 3] == 256 * k for r, f, k, _ in firsts)


def test_long_contexts_get_the_splits_of_a_ragged_batch():
    pos = [8000, 100, 100, 100, 4000, 100, 100, 100]
    rows = np.array([[i, p, i, 0] for i, p in enumerate(pos)], dtype=np.int32)
    items, _ = tuned.balanced_items(rows, 8)
    splits = {int(r): int(w) >> 8 for r, _, _, w in items if r >= 0}
    assert splits[1] == 1 and splits[0] > splits[4] > 8
    # the longest split is not much longer than the mean of the work per place
    longest = max((p + 1) / splits[i] for i, p in enumerate(pos))
    assert longest < 2.0 * sum(p + 1 for p in pos) / len(items) + tuned.DECODE_MIN_KEYS_PER_SPLIT
    # rows of one length share a block per unit and no more; 64 of them get a split each
    even, _ = tuned.balanced_items(np.array([[i, 2099, i, 0] for i in range(8)], dtype=np.int32), 8)
    assert [int(w) >> 8 for r, _, _, w in even if r >= 0 and w & 255 == 0] == [8] * 8
    even, _ = tuned.balanced_items(np.array([[i, 2099, i, 0] for i in range(16)], dtype=np.int32), 8)
    assert [int(w) >> 8 for r, _, _, w in even if r >= 0 and w & 255 == 0] == [2] * 16
    many, _ = tuned.balanced_items(np.array([[i, 2099, i, 0] for i in range(64)], dtype=np.int32), 8)
    assert len(many) == 256 and (many[:64, 3] == 256).all() and (many[64:, 0] < 0).all()
    # no rows, one row
    assert tuned.balanced_items(rows[:0], 8)[0].shape == (0, 4)
    one, first = tuned.balanced_items(rows[:1], 8)
    assert (one[:, 0] >= 0).sum() == 63 and first[0].tolist() == [0, 0, 63, 0]


# ---------------------------------------------------------------- chunks of the linear recurrences
def test_chunks_are_counted_one_for_one():
    """The records that a step asks for are the chunks of the requests that go in chunks, no more, and never beyond what the
    buffer may grow to."""
    from flambeau_amd.kernels.linear_scan import chunks, most_chunks
    assert chunks([2048], 128, 64) == 32 and chunks([2049], 128, 64) == 33
    assert chunks([1] * 64 + [512], 128, 64) == 8                # (requests that walk have none)
    assert chunks([127, 128, 129], 128, 64) == 2 + 3 and chunks([1, 7], 128, 64) == 0
    rng = random.Random(3)
    for _ in range(2000):
        enough, tokens = rng.choice([64, 128, 192, 256]), rng.randint(1, 4096)
        left, lens = tokens, []
        while left:
            lens.append(min(left, rng.choice([1, rng.randint(1, 300), enough, enough + 1, rng.randint(1, 4096)])))
            left -= lens[-1]
        count = sum(1 for q in lens if q >= enough for _ in range(0, q, 64))
        assert chunks(lens, enough, 64) == count <= most_chunks(tokens, enough, 64)


def test_recurrent_mixers_add_nothing_to_a_recorded_steps_key():
    """What goes in chunks follows from the rows per request, which every recorded step's key holds: a step asks these
    mixers for nothing else, whatever the lengths."""
    from flambeau_amd.parts.base import HostBatch
    from flambeau_amd.parts.linear_recurrence import GatedDelta, GatedLinearAttention, Retention, StateSpace
    for cls in (GatedDelta, GatedLinearAttention, Retention, StateSpace):
        for lens in ([1, 1], [300], [1, 300]):
            assert object.__new__(cls).step_signature(HostBatch([0], lens, [5] * len(lens), [0], sum(lens), 1)) == ()


def test_what_goes_in_chunks_is_what_takes_less_time_so():
    """Sizes of both sides that were measured (us walked, us in chunks), few requests and a full chip, whole chunks and begun ones."""
    from flambeau_amd.kernels.linear_scan import FORMS, chunked_from
    for kind, heads, dim, vdim, lens, walked, in_chunks in [
            ("fixed", 16, 128, 128, [2048], 304, 103), ("written", 32, 128, 64, [2048], 310, 106), ("gated", 32, 128, 128, [2048], 311, 150),
            ("delta", 32, 128, 128, [2048], 355, 189), ("delta", 16, 128, 128, [384], 72, 54), ("gated", 32, 128, 128, [129], 29.1, 30.4),
            ("gated", 4, 128, 64, [193] * 4, 31, 34), ("delta", 64, 64, 64, [257], 38, 46), ("delta", 64, 64, 64, [257] * 16, 272, 493),
            ("delta", 64, 64, 64, [1024] * 16, 991, 1475), ("delta", 64, 64, 128, [256], 48.7, 58.1), ("delta", 16, 128, 128, [256], 50, 46),
            ("fixed", 64, 128, 64, [129] * 64, 684, 904), ("fixed", 64, 128, 128, [512] * 16, 1207, 949),
            ("gated", 64, 128, 64, [193] * 64, 1134, 1606), ("written", 64, 64, 64, [129] * 64, 455, 526)]:
        expected = FORMS[kind].tokens if in_chunks < walked else 0
        assert chunked_from(kind, lens, heads, dim, vdim, 64) == expected, (kind, heads, dim, vdim, lens[0], len(lens))
        assert chunked_from(kind, lens + [1], heads, dim, vdim, 64) == expected       # (a token beside them changes nothing)
    for kind in FORMS:
        assert chunked_from(kind, [1] * 8, 32, 128, 128, 64) == 0
