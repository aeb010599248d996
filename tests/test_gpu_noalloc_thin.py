"""Residuals of an allocation-free run on a thin 3D grid: its partials hold 65536
blocks, which the tiles of arbitrary masks pass on a grid where the plain kernel's
block, as the launch names it, covers 1024 cells.  Bit-equal to the oracle, residuals
within the rounding of their sums."""
import ctypes as C

import numpy as np
import pytest

import oracle
from pskel_amd import _lib as L
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu


def test_residuals_of_a_thin_grid(gpu):
    w = 8 * 65536 + 24  # one row of cells along w: 65539 tiles, 513 blocks of (1, 1024)
    pitch = 256
    s = K.Stencil(K.WEIGHTED_SUM, 3, [(0, -1, 0), (0, 0, 0), (0, 1, 0)], weights=[0.25, 0.5, 0.25],
                  boundary=K.BOUNDARY_HALO, halo_value=0.5)
    a = inputs.uniform(12, 0, w).reshape(1, w, 1)
    n = 3
    buf = np.zeros((w, pitch), np.float32)
    buf[:, 0] = a[0, :, 0]
    gd = L.GridDesc()
    gd.ndim, gd.storage, gd.rounding = 3, api._STORAGE["f32"], L.ROUND_NEAREST
    gd.height, gd.width, gd.depth = 1, w, 1
    cfg = api.make_cfg("tuned", block=(1, 1024), residual_every=1)
    d = s.desc()
    res = (C.c_double * n)()
    st = L.RunStats()
    st.residuals = C.cast(res, C.POINTER(C.c_double))
    st.residual_capacity = n
    lib, ptrs = L.lib(), []
    try:
        for _ in range(2):
            p = C.c_void_p()
            L.check(lib.pskel_device_alloc(buf.nbytes, C.byref(p)))
            ptrs.append(p)
            L.check(lib.pskel_memcpy(p, buf.ctypes.data, buf.nbytes, 1))
        L.check(lib.pskel_run_iterative_noalloc(C.byref(gd), ptrs[0], ptrs[1], pitch, C.byref(d), n, C.byref(cfg),
                                                C.byref(st)))
        L.check(lib.pskel_device_synchronize())
        L.check(lib.pskel_memcpy(buf.ctypes.data, ptrs[1], buf.nbytes, 0))
    finally:
        for p in ptrs:
            lib.pskel_device_free(p)
    want, wres = oracle.run_3d(s, a, n, residual_every=1)
    assert np.array_equal(buf[:, 0].view(np.uint32), want[0, :, 0].view(np.uint32))
    assert st.residual_count == n
    np.testing.assert_allclose(list(res), wres, rtol=1e-12, atol=0)
