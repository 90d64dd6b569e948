"""The rounds of a counting collection that stay in one block: lists that fit
its LDS, lists that outgrow what the collections before let expect (512
entries and more), the shallowest trees.  A marking collection behind it finds
nothing left, and the scene reads as the oracle's."""
import numpy as np
import pytest

import oracle_py
import svdag_py


@pytest.mark.gpu
@pytest.mark.parametrize("levels,bits,small,large", [
    (4, 4, 2.0, 6.0), (5, 0, 2.0, 12.0), (9, 8, 1.5, 60.0), (11, 4, 3.0, 200.0), (14, 8, 0.6, 60.0)])
def test_rounds_in_one_block(levels, bits, small, large):
    g = svdag_py.MyGPUHashDAG(levels, bits)
    o = oracle_py.OracleDag(levels, bits)
    s = float(1 << levels)
    rng = np.random.default_rng(levels)
    mats = 3 if bits else 1

    def edit(kind, c, r):
        m = int(rng.integers(0, mats)) if kind in (svdag_py.SPHERE_ADD, svdag_py.BOX_ADD) else 0
        g.edit(kind, m, tuple(c), r)
        o.edit(kind, m, tuple(c), r)

    c = np.array([s / 2, s / 2, s / 2])
    edit(svdag_py.SPHERE_ADD, c, large)
    freed = []
    # small edits first, so that little is expected of the large one's rounds
    for k, r in enumerate([small, small, small * 1.3, large, small, large * 0.9]):
        print(f"[case] release levels={levels} bits={bits} r={r}", flush=True)
        kind = svdag_py.SPHERE_REMOVE if k % 2 else svdag_py.BOX_ADD
        edit(kind, c + rng.uniform(-1, 1, 3) * large / 3, r)
        st = g.garbage_collect()
        freed.append(int(st.items_freed))
        assert st.marked == 0
        check = g.garbage_collect(mark=True)
        assert check.items_freed == 0 and check.items_live == st.items_live
    assert max(freed) > 0
    if levels >= 9:  # more than two of the block's lists
        assert max(freed) > 2 * 512
    pts = rng.integers(0, 1 << levels, (4000, 3)).astype(np.uint32)
    assert np.array_equal(g.query(pts), o.query(pts))
    g.close()


@pytest.mark.gpu
def test_a_round_past_the_list_leaves_the_rest_to_marking():
    # More than 2^21 leaves (the least a round's list holds) die at once: the
    # blocks of the round that overflows the list stop, and the collection
    # marks instead.
    levels = 10
    rng = np.random.default_rng(3)
    noise = np.where(rng.random((512,) * 3, np.float32) < 0.5, np.uint8(0), np.uint8(0xFF))
    g = svdag_py.MyGPUHashDAG(levels, 0, expected_items=1 << 22)
    print("[case] release of more leaves than the list holds", flush=True)
    g.build_voxels(noise)
    for copy in (False, True):  # 2^21 leaves fit, the copy's are too many
        if copy:
            g.build_voxels(noise)
            src = (301.0, 303.0, 202.0)
            assert g.edit(svdag_py.COPY, 0, src, 60.0, src, (760.0, 760.0, 760.0)).applied
        g.garbage_collect(mark=True)  # counts that hold, whatever grew during the build
        g.build_voxels(noise[:64, :64, :64])
        st = g.garbage_collect()
        assert st.marked == copy and st.items_freed > 1 << 21
        assert g.garbage_collect(mark=True).items_freed == 0
    want = svdag_py.MyGPUHashDAG(levels, 0)
    want.build_voxels(noise[:64, :64, :64])
    assert g.canonical() == want.canonical()
    want.close()
    g.close()
