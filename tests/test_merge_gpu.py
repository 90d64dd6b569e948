"""The merge kernels (one lane per item, LDS collapse of duplicates, LDS sums
of child references) at the sizes where they change behaviour: levels of less
than a block, several blocks, chains that grow, contents that repeat."""
import numpy as np
import pytest

import oracle_py
import svdag_py


def _noise(side, rng, fill, mats):
    vox = np.full((side,) * 3, 0xFF, np.uint8)
    pick = rng.uniform(size=(side,) * 3) < fill
    vox[pick] = rng.choice(mats, int(pick.sum()))
    return vox


@pytest.mark.gpu
@pytest.mark.parametrize("bits,lanes,grid_log2,pattern", [
    (0, 4, 4, "noise"), (4, 32, 5, "noise"), (8, 0, 6, "noise"),
    (0, 0, 6, "noise"), (4, 0, 7, "repeat"), (8, 16, 6, "repeat"), (4, 8, 2, "noise")])
def test_merge_matches_oracle_and_counts_references(bits, lanes, grid_log2, pattern):
    levels, side = 8, 1 << grid_log2
    rng = np.random.default_rng(100 * bits + 10 * grid_log2 + lanes)
    mats = [0] if bits == 0 else list(range(1, min(15, (1 << bits) - 2)))
    if pattern == "noise":
        vox = _noise(side, rng, 0.3, mats)
    else:  # sixteen different bricks over and over
        bricks = [_noise(8, rng, 0.4, mats) for _ in range(16)]
        vox = np.empty((side,) * 3, np.uint8)
        for x in range(0, side, 8):
            for y in range(0, side, 8):
                for z in range(0, side, 8):
                    vox[x:x + 8, y:y + 8, z:z + 8] = bricks[rng.integers(16)]
    # Tables of 64 buckets: chains grow while the level is inserted.
    g = svdag_py.MyGPUHashDAG(levels, bits, group_size=lanes, expected_items=64, arena_slabs=1 << 17)
    o = oracle_py.OracleDag(levels, bits)
    print(f"[case] merge bits={bits} lanes={lanes} side={side} {pattern}", flush=True)
    g.build_voxels(vox)
    full = np.full((1 << levels,) * 3, 0xFF, np.uint8)
    full[:side, :side, :side] = vox
    oracle_py.build_dense(o, full)
    assert g.canonical() == o.canonical()
    edits = [(svdag_py.BOX_ADD, mats[0], (100.0, 90.0, 120.0), 37.0), (svdag_py.SPHERE_ADD, mats[-1], (60.0, 60.0, 60.0), 30.0),
             (svdag_py.BOX_REMOVE, 0, (110.0, 90.0, 100.0), 9.0), (svdag_py.PAINT, mats[-1], (100.0, 70.0, 120.0), 25.0)]
    g.edit_batch(edits)
    for kind, mat, c, r in edits:
        o.edit(kind, mat, c, r)
    assert g.canonical() == o.canonical()
    # A marking collection right after a counting one frees nothing: the
    # counts the merge kept are those of the stored items.
    counted = g.garbage_collect()
    marked = g.garbage_collect(mark=True)
    assert counted.marked == 0 and marked.items_freed == 0
    assert counted.items_live == marked.items_live
    assert g.canonical() == o.canonical()
    g.close()


@pytest.mark.gpu
def test_levels_around_the_one_block_limit_match_oracle():
    # Levels of 1025 to 2048 items among those one block takes (its threads
    # loop there), from one copy and from a wave of paints; and a wave of one
    # tiny edit.
    levels, side = 8, 256
    rng = np.random.default_rng(77)
    vox = np.full((side,) * 3, 0xFF, np.uint8)
    cells = [(x, y, z) for x in range(4) for y in range(2) for z in range(2)][:14]
    for cx, cy, cz in cells:
        c = tuple(64 * v + 8 for v in (cx, cy, cz))
        vox[c[0]:c[0] + 48, c[1]:c[1] + 48, c[2]:c[2] + 48] = _noise(48, rng, 0.4, [1, 2, 3, 4])
    vox[:96, 160:, 160:] = _noise(96, rng, 0.4, [5, 6])
    g = svdag_py.MyGPUHashDAG(levels, 4)
    o = oracle_py.OracleDag(levels, 4)
    g.build_voxels(vox)
    oracle_py.build_dense(o, vox)
    paints = [(svdag_py.PAINT, 5 + i, (64.0 * cx + 32, 64.0 * cy + 32, 64.0 * cz + 32), 16.0)
              for i, (cx, cy, cz) in enumerate(cells[:10])]
    copy = (svdag_py.COPY, 0, (48.0, 208.0, 208.0), 44.0, (48.0, 208.0, 208.0), (180.0, 180.0, 70.0))
    tiny = (svdag_py.SPHERE_ADD, 7, (200.0, 20.0, 20.0), 0.4)
    big = [(svdag_py.PAINT, 15, (64.0 * cx + 32, 64.0 * cy + 32, 64.0 * cz + 32), 23.0) for cx, cy, cz in cells]
    per_level = []
    for batch in (paints, [copy], [tiny], big):
        stats, _ = g.edit_batch(batch)
        per_level.append(np.sum([list(s.svo_items) for s in stats], axis=0))
        for e in batch:
            o.edit(*e)
        assert g.canonical() == o.canonical()
    assert any(((n > 1024) & (n <= 2048)).any() for n in per_level)
    st = g.garbage_collect()
    assert st.marked == 0 and g.garbage_collect(mark=True).items_freed == 0
    g.close()


def _corner_scene(levels):
    """Voxels around the lattice corners that are odd multiples of 16: below
    each corner up to its sides, above it only from 10 voxels on.  All eight
    16-voxel cells around a corner hold voxels, but only the lower four of the
    8-voxel cells do."""
    side = 1 << levels
    rng = np.random.default_rng(5)
    vox = _noise(side, rng, 0.6, [1, 2, 3, 4])
    y = np.arange(side) % 32  # the corner is at 16
    vox[:, ~(((y >= 11) & (y < 16)) | ((y >= 26) & (y < 30))), :] = 0xFF
    return vox


@pytest.mark.gpu
@pytest.mark.parametrize("bits,lanes", [(4, 0), (8, 4)])
def test_a_large_level_above_a_small_one_matches_oracle(bits, lanes):
    # 200 small paints (the tool that leaves empty children alone), each with
    # 8 items on level 4 and 4 on level 5, in one wave split at level 4: one
    # block takes both levels, the lower one with an item per thread and the
    # upper one through the workspace, where it reads what the lower one left.
    levels, edits = 8, 200
    vox = _corner_scene(levels)
    g = svdag_py.MyGPUHashDAG(levels, bits, group_size=lanes)
    o = oracle_py.OracleDag(levels, bits)
    g.build_voxels(vox)
    oracle_py.build_dense(o, vox)
    rng = np.random.default_rng(9)
    corners = np.stack(np.meshgrid(*[np.arange(16, 1 << levels, 32)] * 3, indexing="ij"), -1).reshape(-1, 3)
    print(f"[case] large above small bits={bits} lanes={lanes}", flush=True)
    for rep in range(3):  # results left by one batch would show in the next
        at = corners[rng.permutation(len(corners))[:edits]]
        batch = [(svdag_py.PAINT, 5 + rep, tuple(map(float, c)), 1.6 + 0.4 * rep) for c in at]
        stats, _ = g.edit_batch(batch)
        items = np.sum([list(s.svo_items) for s in stats], axis=0)
        # The host's bound of both levels is 8 items an edit (at most 2048).
        assert items[4] > 1024 and 0 < items[5] <= 1024 and 8 * edits <= 2048
        for e in batch:
            o.edit(*e)
        assert g.canonical() == o.canonical()
    st = g.garbage_collect()
    assert st.marked == 0 and g.garbage_collect(mark=True).items_freed == 0
    g.close()


@pytest.mark.gpu
def test_leaves_with_the_words_of_stored_nodes_get_their_own_items():
    # At no material bits a leaf's two words can be those of a node with one
    # child; a merge finds the node, which has another role, and must store
    # the leaf beside it, once.
    levels, side = 8, 64
    rng = np.random.default_rng(4)
    vox = np.full((side,) * 3, 0xFF, np.uint8)
    for at in rng.choice(512, 60, replace=False):  # one leaf in a cell of 8: nodes of one child
        x, y, z = (8 * v for v in (at // 64, at // 8 % 8, at % 8))
        vox[x:x + 4, y:y + 4, z:z + 4][rng.random((4, 4, 4)) < 0.4] = 0
    g = svdag_py.MyGPUHashDAG(levels, 0)
    g.build_voxels(vox)
    rec, p, twins = g.export_records(), 4, []
    while p < len(rec):
        size = int(rec[p + 2])
        if rec[p] == levels - 3 and size == 2:
            twins.append(int(rec[p + 3]) | int(rec[p + 4]) << 32)
        p += 3 + size
    assert len(twins) > 30
    both = np.full((2 * side,) * 3, 0xFF, np.uint8)
    both[:side, :side, :side] = vox
    for k, bits in enumerate(twins * 2):  # each twice, as a leaf of the other half
        x, y, z = side + 8 * (k % 8), side + 8 * (k // 8 % 8), side + 8 * (k // 64)
        for b in range(64):
            if bits >> b & 1:
                both[x + (b >> 5 & 1) * 2 + (b >> 2 & 1), y + (b >> 4 & 1) * 2 + (b >> 1 & 1),
                     z + (b >> 3 & 1) * 2 + (b & 1)] = 0
    print("[case] leaves equal to nodes", flush=True)
    o = oracle_py.OracleDag(levels, 0)
    full = np.full((1 << levels,) * 3, 0xFF, np.uint8)
    full[:2 * side, :2 * side, :2 * side] = both
    oracle_py.build_dense(o, full)
    for again in range(2):
        g.build_voxels(both)
        assert g.canonical() == o.canonical()
        st = g.garbage_collect()
        marked = g.garbage_collect(mark=True)
        assert marked.items_freed == 0 and marked.items_live == st.items_live
        live = st.items_live if not again else live
        assert st.items_live == live
    g.close()
