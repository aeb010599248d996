"""Fused 2D sweeps on a caller's buffers (pskel_run_iterative_noalloc) leave the
padding of its rows alone, whatever the width's remainder; the cells equal the
oracle's.  An odd number of sweeps ends in `out` without a copy of the buffers."""
import ctypes as C

import numpy as np
import pytest

import oracle
from pskel_amd import _lib as L
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu


def _check(s, a, b, n, k):
    h, w = a.shape
    pitch = -(-w * a.itemsize // 1024) * 1024 // a.itemsize + 1024 // a.itemsize
    pad = (77, 99)
    bufs = []
    for host, value in ((a, pad[0]), (b, pad[1])):
        m = np.full((h, pitch), value, a.dtype)
        m[:, :w] = host
        bufs.append(m)
    gd = L.GridDesc()
    gd.ndim, gd.storage = 2, api._STORAGE["u8" if a.dtype == np.uint8 else "f32"]
    gd.height, gd.width, gd.depth = h, w, 1
    gd.rounding = L.ROUND_NEAREST
    cfg = api.make_cfg("tuned", time_tile=k)
    d = s.desc()
    lib, ptrs = L.lib(), []
    try:
        for m in bufs:
            p = C.c_void_p()
            L.check(lib.pskel_device_alloc(m.nbytes, C.byref(p)))
            ptrs.append(p)
            L.check(lib.pskel_memcpy(p, m.ctypes.data, m.nbytes, 1))
        L.check(lib.pskel_run_iterative_noalloc(C.byref(gd), ptrs[0], ptrs[1], pitch, C.byref(d), n, C.byref(cfg), None))
        L.check(lib.pskel_device_synchronize())
        for m, p in zip(bufs, ptrs):
            L.check(lib.pskel_memcpy(m.ctypes.data, p, m.nbytes, 0))
    finally:
        for p in ptrs:
            lib.pskel_device_free(p)
    assert np.array_equal(bufs[1][:, :w], oracle.run_2d(s, a, n, out=b)), (w, n)
    for m, value in zip(bufs, pad):
        assert (m[:, w:] == value).all(), (w, n)


@pytest.mark.parametrize("name", ["jacobi2d", "diffusion9"])
@pytest.mark.parametrize("width", [9, 10, 11, 12, 255, 256, 257, 258, 259, 1021])
def test_f32_padding(gpu, name, width):
    a = inputs.uniform(width, 0, 70 * width).reshape(70, width)
    b = a.copy()
    b[0, :], b[-1, :], b[:, 0], b[:, -1] = 3.0, -2.0, 0.5, 7.0
    for n in (1, 5, 17):
        _check(getattr(K, name)(), a, b, n, 4)


@pytest.mark.parametrize("width", list(range(1, 34)) + [47, 48, 50, 1503, 2047, 2048, 2049, 2063, 2064, 2066])
def test_life_padding(gpu, width):
    a = (inputs.uniform(width, 0, 40 * width).reshape(40, width) < np.float32(0.35)).astype(np.uint8)
    b = a.copy()
    b[0, :], b[-1, :], b[:, 0], b[:, -1] = 1 - a[0, :], 1 - a[-1, :], 1 - a[:, 0], 1 - a[:, -1]
    for n in (1, 5, 17):
        _check(K.life(), a, b, n, 8)
