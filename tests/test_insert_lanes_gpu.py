"""Bulk inserts (one lane per item for every variant): more segments than one
launch takes, ragged and empty ones, items of 1 to 18 words, equal items,
chains that grow from a handful of buckets."""
import numpy as np
import pytest

import svdag_py


@pytest.mark.gpu
@pytest.mark.parametrize("variant,lo,hi,buckets", [(0, 2, 9, 3), (16, 1, 18, 40), (32, 2, 18, 1), (4, 3, 10, 500), (8, 18, 18, 7)])
def test_bulk_insert_stores_every_item_once(variant, lo, hi, buckets):
    rng = np.random.default_rng(variant * 100 + hi)
    groups = []
    for k in range(45):
        s = lo + k % (hi - lo + 1)
        n = int(rng.choice([0, 1, 63, 64, 255, 256, 257, 700]))
        arr = rng.integers(0, 1 << 32, size=(n, s), dtype=np.uint64).astype(np.uint32)
        if n > 64 and k % 3 == 0:
            arr[1:40] = arr[0]  # equal items: a multiset
        groups.append((s, arr))
    words, segs, n = svdag_py.make_segments(groups)
    sizes = range(lo, hi + 1)
    per = [sum(len(a) for t, a in groups if t == s) for s in sizes]
    print(f"[case] insert variant={variant} sizes {lo}..{hi} buckets={buckets} items={n}", flush=True)
    hs = svdag_py.HashSet(lo, hi, [buckets] * len(per), [2 * p for p in per])
    wdev = svdag_py.DeviceBuffer.from_array(words)
    odev = svdag_py.DeviceBuffer(4 * n)
    hs.add_dev(wdev, segs, odev, variant)
    ptrs = odev.to_array(np.uint32, n)
    assert (ptrs != svdag_py.NOT_FOUND).all()
    for s in sizes:
        mine = np.concatenate([ptrs[g.out_offset:g.out_offset + g.count] for g in segs if g.item_words == s] + [ptrs[:0]])
        want = np.concatenate([a for t, a in groups if t == s] + [np.zeros((0, s), np.uint32)])
        assert len(np.unique(mine)) == len(mine)
        if len(mine):
            assert np.array_equal(hs.read(s, mine), want)
    hs.find_dev(wdev, segs, odev, 16)
    assert (odev.to_array(np.uint32, n) != svdag_py.NOT_FOUND).all()
    hs.close()
