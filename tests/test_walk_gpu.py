"""The ray walk where it branches: the shallowest and the deepest stack, images
that end inside a tile, rays with a zero direction component (infinite
inverses), an origin far outside, filled nodes that end an occlusion ray."""
import numpy as np
import pytest

import oracle_py
import svdag_py


def _scene(levels, bits):
    g = svdag_py.MyGPUHashDAG(levels, bits)
    o = oracle_py.OracleDag(levels, bits)
    s = float(1 << levels)
    m = [1, 2, 3] if bits else [0, 0, 0]
    r = min(s / 5, 40.0)
    edits = [(svdag_py.BOX_ADD, m[0], (s / 2, s / 2, s / 2), r), (svdag_py.SPHERE_REMOVE, 0, (s / 2 + r, s / 2, s / 2), r * 0.7),
             (svdag_py.SPHERE_ADD, m[1], (s / 2 - r, s / 2 + r, s / 2), r * 0.5),
             (svdag_py.BOX_ADD, m[2], (s / 2, s / 2 - 1.2 * r, s / 2), 0.3 * r)]
    for kind, mat, c, rad in edits:
        g.edit(kind, mat, c, rad)
        o.edit(kind, mat, c, rad)
    return g, o, s, r


def _same_hits(a, b):
    for f in ("x", "y", "z", "material"):
        assert np.array_equal(a[f], b[f]), f
    for f in ("t", "px", "py", "pz"):
        assert np.array_equal(a[f], b[f], equal_nan=True), f


@pytest.mark.gpu
@pytest.mark.parametrize("levels,bits,w,h,view", [
    (4, 0, 1, 1, "corner"), (5, 8, 17, 9, "corner"), (9, 4, 64, 32, "axis"), (9, 0, 33, 65, "axis"),
    (20, 4, 40, 24, "corner"), (20, 8, 16, 16, "axis"), (10, 4, 30, 50, "far")])
def test_walk_matches_oracle(levels, bits, w, h, view):
    g, o, s, r = _scene(levels, bits)
    c = np.array([s / 2, s / 2, s / 2])
    pos = {"corner": c + r * np.array([2.5, 2.1, 1.7]), "axis": c + np.array([0.0, 0.0, 3.0 * r]),
           "far": c + 1e6 * np.array([0.5, 0.4, 0.3])}[view]
    fov = 1e-2 if view == "far" else 50.0
    rot = svdag_py.look_at(pos, c)
    args = (tuple(pos), rot, fov, (0.0,) * 3, (s,) * 3, w, h)
    print(f"[case] walk levels={levels} bits={bits} {w}x{h} {view}", flush=True)
    hits, _ = g.trace(*args)
    want = o.trace(*args)
    _same_hits(hits, want)
    assert w * h == 1 or (hits["material"] != svdag_py.NOT_FOUND).any()
    for length in (4.0, float("inf")):
        sun, _ = g.trace_shadows(0.25)
        ao, _ = g.trace_ambient_occlusion(2, 0.25, length, 5)
        osun, oao = o.shade(*args, bias=0.25, ao_samples=2, ao_length=length, seed=5)
        assert np.array_equal(sun, osun) and np.array_equal(ao, oao)
    g.close()


@pytest.mark.gpu
def test_imported_full_flags_do_not_end_occlusion_rays():
    # An imported node may carry the full flag over children that are not all
    # filled; rays pass through its empty parts all the same.
    levels, bits, w, h = 8, 4, 96, 64
    g, _, s, r = _scene(levels, bits)
    _, _, dump = g.canonical(dump=True)
    forged, p, changed = dump.copy(), 0, 0
    for level in range(levels - 2, -1, -1):
        count, p = int(dump[p + 1]), p + 2
        for _ in range(count):
            if level < levels - 2 and dump[p + 1] & 0xFF != 0xFF:
                forged[p + 1] |= 0x100
                changed += 1
            p += 1 + int(dump[p])
    assert changed > 100
    f = svdag_py.MyGPUHashDAG(levels, bits)
    f.import_canonical(forged)
    c = np.array([s / 2, s / 2, s / 2])
    pos = c + r * np.array([2.5, 2.1, 1.7])
    args = (tuple(pos), svdag_py.look_at(pos, c), 50.0, (0.0,) * 3, (s,) * 3, w, h)
    palette = np.linspace(0.1, 0.9, 3 * 16).reshape(16, 3)
    out = []
    for d in (g, f):
        hits, _ = d.trace(*args)
        sun, _ = d.trace_shadows(0.25)
        ao, _ = d.trace_ambient_occlusion(4, 0.25, 30.0, 5)
        d.trace_colors(palette)
        path, _, _ = d.trace_path_tracing(palette, samples=2, depth=3)
        out.append((hits.view(np.uint32), sun, ao, path))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    assert (out[0][1] > 0).any() and ((out[0][2] > 0) & (out[0][2] < 1)).any()
    g.close()
    f.close()
