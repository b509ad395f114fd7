"""Key-split prefill attention: how a call's keys are dealt to workgroups (host
arithmetic, no GPU)."""
import ctypes
import random

import numpy as np


def _chunks(b, sq, sk, hq, hkv, d, causal, window):
    """(queries per tile, keys per tile, merged [tiles], first and end key tile
    [tiles, chunks]) of a call, or None where its keys are not split."""
    from torchplusplus_amd._native import lib
    dims, i64 = (ctypes.c_int32 * 4)(), ctypes.c_int64
    shape = [*map(i64, (b, sq, sk, hq, hkv, d)), int(causal), *window]
    assert lib().tpp_attn_prefill_chunks(*shape, dims, None, i64(0)) == 0
    ql, kt, tiles, chunks = dims
    if not chunks:
        return None
    out = np.full((tiles, 1 + 2 * chunks), -1, dtype=np.int32)
    assert lib().tpp_attn_prefill_chunks(*shape, dims, ctypes.c_void_p(out.ctypes.data), i64(out.size)) == 0
    return ql, kt, out[:, 0], out[:, 1::2], out[:, 2::2]


def _calls():
    """Lengths around the tiles, windows on both sides, every group form."""
    heads = [(16, 8), (8, 8), (8, 4), (24, 8), (24, 6), (4, 4), (16, 2), (3, 1)]
    sizes = [1, 17, 31, 33, 64, 65, 100, 177, 260, 300, 340, 400, 521, 700, 784, 900, 1000, 1999, 2500]
    rng = random.Random(7)
    for sq in sizes:
        for extra in (0, 3, 200, 300, 2318, -7):
            for d in (64, 128):
                for left in (-1, 0, 33, 127, 199, 200, 255, 511, 601, 700, 1000, 1392):
                    hq, hkv = rng.choice(heads)
                    right = rng.choice([-1, 0, 0, 0, 50, 78])
                    yield rng.choice([1, 1, 2]), sq, max(1, sq + extra), hq, hkv, d, right == 0, (left, right)
    for _ in range(6000):
        sq = int(2 ** rng.uniform(0, 12))
        hq, hkv = rng.choice(heads)
        right = rng.choice([-1, 0, 0, rng.randrange(1, 2000)])
        yield (rng.choice([1, 1, 2, 4]), sq, max(1, sq + rng.choice([0, 0, rng.randrange(-50, 6000)])), hq, hkv,
               rng.choice([64, 128]), right == 0, (rng.choice([-1, rng.randrange(2000)]), right))


# calls that dealt a query tile fewer chunks than its keys need
NAMED = [(1, 300, 300, 16, 8, 64, True, (200, 0)), (1, 700, 700, 16, 8, 64, True, (200, 0)),
         (1, 400, 400, 8, 8, 128, True, (199, 0)), (1, 900, 1100, 8, 4, 128, True, (1000, 0)),
         (1, 784, 784, 24, 8, 64, False, (601, 77)), (1, 177, 2495, 24, 6, 64, False, (1392, 78)),
         (1, 521, 821, 4, 4, 128, True, (700, 0)), (1, 260, 260, 16, 8, 128, False, (199, 50))]


def _visible_tiles(sq, sk, ql, kt, window):
    """First and end tile of the keys that each query tile sees (empty: both
    equal), one query row at a time: key j is visible from query i iff
    -left <= j - (i + sk - sq) <= right."""
    left, right = window
    pos = np.arange(sq) + sk - sq
    lo = np.maximum(pos - left, 0) if left >= 0 else np.zeros(sq, dtype=np.int64)
    hi = np.minimum(pos + right + 1, sk) if right >= 0 else np.full(sq, sk)
    some = hi > lo
    tile = np.arange(sq) // ql
    first = np.full(tile[-1] + 1, 1 << 30)
    end = np.zeros(tile[-1] + 1, dtype=np.int64)
    np.minimum.at(first, tile[some], lo[some] // kt)
    np.maximum.at(end, tile[some], (hi[some] + kt - 1) // kt)
    return np.where(end > 0, first, 0), end


def test_every_visible_key_is_in_one_chunk():
    """The chunks of a query tile follow one another without a gap, from no
    later than its first visible key to no earlier than its last."""
    several = 0
    for call in NAMED + list(_calls()):
        plan = _chunks(*call)
        if plan is None:
            continue
        (_, sq, sk, _, _, _, causal, window), (ql, kt, merged, first, end) = call, plan
        want_first, want_end = _visible_tiles(sq, sk, ql, kt, (window[0], 0 if causal else window[1]))
        seen = want_end > 0
        several += first.shape[1] > 1
        ran = np.arange(first.shape[1])[None, :] < merged[:, None]
        assert (merged[seen] > 0).all(), call
        last = np.take_along_axis(end, np.maximum(merged - 1, 0)[:, None], 1)[:, 0]
        assert (first[:, 0] <= want_first)[seen].all() and (last >= want_end)[seen].all(), call
        assert (first[:, 1:] == end[:, :-1])[ran[:, 1:]].all(), call
        # no chunk longer than a full one (its time is what the plan counted)
        assert ((end - first).max(axis=1) <= (end - first)[:, 0])[merged > 1].all(), call
    assert several > 500


def test_merge_reads_only_chunks_that_were_written():
    split = 0
    for call in NAMED + list(_calls()):
        plan = _chunks(*call)
        if plan is None:
            continue
        _, _, merged, first, end = plan
        split += 1
        assert (merged <= first.shape[1]).all(), call
        ran = np.arange(first.shape[1])[None, :] < merged[:, None]
        assert (first < end)[ran].all() and not (first < end)[~ran].any(), call
    assert split > 2000
