"""Frame results that the kernels store in pinned host memory themselves equal
the copied ones, which the oracle covers: whole and cut tiles, the smallest
stack, a result inside a larger buffer, one that a hit record's halves do not
align to, and nothing written beside it."""
import ctypes

import numpy as np
import pytest

import svdag_py
from test_walk_gpu import _scene


def _pinned(nbytes, offset):
    """(pointer, all of a pinned buffer, the part of it that a pass may write)"""
    p = ctypes.c_void_p()
    size = nbytes + 512
    # the library's own runtime, found through its dependencies
    assert svdag_py.lib().hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(size), ctypes.c_uint(0)) == 0
    a = np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_uint8)), (size,))
    a[:] = 0xA5
    return p, a, a[128 + offset: 128 + offset + nbytes]


def _passes(g, cam, w, h, palette, into, timed):
    """Every pass, its result in into(name, bytes); gpu_ms asked for or not."""
    lib, n = svdag_py.lib(), w * h
    ms = ctypes.c_float(0)
    pms = ctypes.byref(ms) if timed else None
    got = {}

    def run(name, size, call):
        buf = into(name, n * size)
        svdag_py.check(call(buf.ctypes.data_as(ctypes.c_void_p)))
        got[name] = buf.copy()

    pal = palette.ctypes.data_as(ctypes.c_void_p)
    u32, u64, f32 = ctypes.c_uint32, ctypes.c_uint64, ctypes.c_float
    run("hits", 32, lambda p: lib.svdag_trace_primary(g.h, ctypes.byref(cam), w, h, p, pms))
    run("ao", 4, lambda p: lib.svdag_trace_ambient_occlusion(g.h, u32(2), f32(0.25), f32(8.0), u64(5), p, pms))
    if w % 8 == 0 and h % 8 == 0:
        run("blur", 4, lambda p: lib.svdag_blur_ambient_occlusion(g.h, p, pms))
    run("sun", 4, lambda p: lib.svdag_trace_shadows(g.h, f32(0.25), p, pms))
    run("colors", 4, lambda p: lib.svdag_trace_colors(g.h, pal, u32(len(palette)), p, pms))
    light = svdag_py.Lighting(1, 1, 0.0, 0.8)
    run("light", 4, lambda p: lib.svdag_trace_lighting(g.h, ctypes.byref(light), p, pms))
    path = svdag_py.PathTracing(1.0, 2, 3, 0, 11, 0, 0)
    run("path", 4, lambda p: lib.svdag_trace_path_tracing(g.h, ctypes.byref(path), pal, u32(len(palette)), p, None, pms))
    return got


@pytest.mark.gpu
@pytest.mark.parametrize("levels,w,h,offset", [
    (4, 8, 8, 0), (5, 1, 1, 0), (9, 64, 40, 0), (9, 71, 37, 16), (10, 40, 24, 4), (14, 250, 130, 0)])
def test_results_stored_by_the_kernels(levels, w, h, offset):
    g, _, s, r = _scene(levels, 4)
    c = np.array([s / 2, s / 2, s / 2])
    pos = c + r * np.array([2.5, 2.1, 1.7])
    cam = g._camera(tuple(pos), svdag_py.look_at(pos, c), 50.0, (0.0,) * 3, (s,) * 3)
    palette = np.random.default_rng(3).uniform(0.2, 0.9, (16, 3)).astype(np.float32)
    print(f"[case] frame results levels={levels} {w}x{h} offset={offset}", flush=True)
    want = _passes(g, cam, w, h, palette, lambda _, n: np.zeros(n, np.uint8), True)
    kept = {}

    def pinned(name, n):
        if name not in kept:
            kept[name] = _pinned(n, offset)
        kept[name][2][:] = 0xA5
        return kept[name][2]

    got = _passes(g, cam, w, h, palette, pinned, False)
    again = _passes(g, cam, w, h, palette, pinned, True)  # the same buffers, copied
    for name, v in want.items():
        assert np.array_equal(got[name], v), name
        assert np.array_equal(again[name], v), name
    at = 128 + offset
    for p, whole, part in kept.values():
        assert (whole[:at] == 0xA5).all() and (whole[at + part.size:] == 0xA5).all()
    g.close()
    for p, _, _ in kept.values():
        svdag_py.lib().hipHostFree(p)
