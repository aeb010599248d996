"""Every tile shape that is built of the 2D kernels, named by the test (a run's plan
picks it by the grid's size), bit-equal to the oracle on ragged grids with distinct
rings: register tiles with and without residual partials and with the state before
the last sweep, life tiles, the register march and the LDS tile.  The partials are
FP64 sums over the same cells in another order: within 1e-12."""
import ctypes as C

import numpy as np
import pytest

import oracle
import shapes
from pskel_amd import _lib as L
from pskel_amd import inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu

NAMES = {shapes.J5: "jacobi2d", shapes.BOX9: "diffusion9", shapes.CLOUD: "cloudsim"}
RT = ([(shapes.J5, r, nw) for r, nw in ((2, 16), (4, 8), (4, 16), (8, 8))] +
      [(shapes.BOX9, r, nw) for r, nw in ((2, 8), (2, 16), (4, 8), (4, 16))] +
      [(shapes.CLOUD, r, nw) for r, nw in ((2, 8), (2, 16), (4, 8))])
LT = [(2, 8), (2, 16), (4, 16), (8, 8), (8, 16)]


class _Buffers:
    """device buffers of pitched rows, freed together"""

    def __init__(self):
        self.ptrs = []

    def new(self, host=None, nbytes=0):
        p = C.c_void_p()
        L.check(L.lib().pskel_device_alloc(host.nbytes if host is not None else nbytes, C.byref(p)))
        self.ptrs.append(p)
        if host is not None:
            L.check(L.lib().pskel_memcpy(p, host.ctypes.data, host.nbytes, 1))
        return p.value

    def read(self, p, like):
        out = np.empty_like(like)
        L.check(L.lib().pskel_memcpy(out.ctypes.data, p, out.nbytes, 0))
        return out

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        for p in self.ptrs:
            L.lib().pskel_device_free(p)


def _pitched(a):
    pitch = -(-a.shape[1] * a.itemsize // 1024) * 1024 // a.itemsize
    m = np.zeros((a.shape[0], pitch), a.dtype)
    m[:, :a.shape[1]] = a
    return m


def _inputs(pattern, shape):
    """state, other buffer, wind fields, state after n sweeps"""
    if pattern == shapes.CLOUD:
        a, wx, wy = inputs.cloudsim_fields(*shape, seed=sum(shape))
        b = a.copy()
        b[0, :], b[-1, :], b[:, 0], b[:, -1] = 3.0, -2.0, 0.5, 7.0
        return a, b, (wx, wy), lambda n: oracle.run_2d_cloud(a, wx, wy, 0.01, n, out=b) if n else a
    u = inputs.uniform(sum(shape), 0, shape[0] * shape[1]).reshape(shape)
    if pattern == shapes.LIFE8:
        a = (u < np.float32(0.35)).astype(np.uint8)
        b = a.copy()
        b[0, :], b[-1, :], b[:, 0], b[:, -1] = 1 - a[0, :], 1 - a[-1, :], 1 - a[:, 0], 1 - a[:, -1]
        s = K.life()
    else:
        a, s = u, getattr(K, NAMES[pattern])()
        b = a.copy()
        b[0, :], b[-1, :], b[:, 0], b[:, -1] = 3.0, -2.0, 0.5, 7.0
    return a, b, None, lambda n: oracle.run_2d(s, a, n, out=b) if n else a


def _job(bufs, pattern, a, b, winds, k, keep=False):
    """the launch as a run issues it: odd k writes the other buffer, even k a spare"""
    j = shapes.Job()
    h, w = a.shape
    am, bm = _pitched(a), _pitched(b)
    spare = am.copy()
    spare[1:-1, 1:w - 1] = 0  # the current state's ring, another interior
    j.src, j.ring = bufs.new(am), bufs.new(bm)
    j.dst = j.ring if k % 2 else bufs.new(spare)
    if keep and k > 1:  # the state before the last sweep: the buffer of its ring, or any other
        j.prev = bufs.new(np.zeros_like(am)) if k % 2 else j.ring
    j.pitch, j.W, j.H, j.pattern, j.k = am.shape[1], w, h, pattern, k
    if pattern == shapes.CLOUD:
        j.coeff = 0.01
        # the device layout of a field: cell (h, w) in row h
        xm, ym = _pitched(np.ascontiguousarray(winds[0].T)), _pitched(np.ascontiguousarray(winds[1].T))
        j.wx, j.wy, j.xpitch, j.ypitch = bufs.new(xm), bufs.new(ym), xm.shape[1], ym.shape[1]
    elif pattern != shapes.LIFE8:
        d = getattr(K, NAMES[pattern])().desc()
        j.coeff = d.coeff
        for i in range(9):
            j.wt[i] = d.weights[i]
    return j, am


def _same(got, want, what):
    assert np.array_equal(got[:, :want.shape[1]].view(np.uint8), want.view(np.uint8)), what


@pytest.mark.parametrize("pattern,r,nw", RT)
def test_register_tile_shapes(gpu, pattern, r, nw):
    l = shapes.lib()
    rows = r * nw
    for shape in ((rows - 1, 94), (rows, 257), (rows + 1, 523), (3 * rows + 5, 1030)):
        a, b, winds, state = _inputs(pattern, shape)
        for k in (1, 2, 3, min(7, rows // 2 - 1), min(32, rows // 2 - 2)):
            for residual, keep in ((False, False), (True, False), (False, True), (True, True)):
                with _Buffers() as bufs:
                    j, am = _job(bufs, pattern, a, b, winds, k, keep)
                    nb = l.shapes_rtile_blocks(shape[1], shape[0], r, nw, k)
                    part = np.full(nb, np.nan)
                    if residual:
                        j.partials = bufs.new(part)
                    assert l.shapes_rtile(C.byref(j), r, nw) == 0, (shape, k)
                    L.check(L.lib().pskel_device_synchronize())
                    want, before = state(k), state(k - 1)
                    _same(bufs.read(j.dst, am), want, (shape, k, residual))
                    if j.prev:
                        _same(bufs.read(j.prev, am), before, (shape, k, residual, "prev"))
                    if residual:
                        total = bufs.read(j.partials, part).sum()
                        d = want.astype(np.float64) - before.astype(np.float64)
                        np.testing.assert_allclose(total, (d * d).sum(), rtol=1e-12, atol=0)


@pytest.mark.parametrize("r,nw", LT)
def test_life_tile_shapes(gpu, r, nw):
    l = shapes.lib()
    rows = r * nw
    for shape in ((rows - 1, 33), (rows, 2049), (rows + 1, 2078), (3 * rows + 5, 4100)):
        a, b, _, state = _inputs(shapes.LIFE8, shape)
        for k in (1, 2, min(7, rows // 2 - 1), min(30, rows // 2 - 2), min(31, rows // 2 - 1)):
            for keep in (False, True):
                with _Buffers() as bufs:
                    j, am = _job(bufs, shapes.LIFE8, a, b, None, k, keep)
                    assert l.shapes_life(C.byref(j), r, nw) == 0, (shape, k)
                    L.check(L.lib().pskel_device_synchronize())
                    _same(bufs.read(j.dst, am), state(k), (shape, k, keep))
                    if j.prev:
                        _same(bufs.read(j.prev, am), state(k - 1), (shape, k, "prev"))


@pytest.mark.parametrize("pattern", [shapes.J5, shapes.BOX9])
def test_march_and_lds_tile_shapes(gpu, pattern):
    l = shapes.lib()
    for shape in ((3, 9), (41, 523), (100, 1021)):
        a, b, _, state = _inputs(pattern, shape)
        for k in (2, 3, 4):
            want = state(k)
            for run, arg in [(l.shapes_march, s) for s in (0, 5, 8, 64)] + [(l.shapes_ttile, y) for y in (8, 16, 32, 64)]:
                with _Buffers() as bufs:
                    j, am = _job(bufs, pattern, a, b, None, k)
                    assert run(C.byref(j), arg) == 0, (shape, k, arg)
                    L.check(L.lib().pskel_device_synchronize())
                    _same(bufs.read(j.dst, am), want, (shape, k, run.__name__, arg))


def test_shapes_that_are_not_built(gpu):
    l = shapes.lib()
    a, b, winds, _ = _inputs(shapes.J5, (40, 300))
    with _Buffers() as bufs:
        j, _ = _job(bufs, shapes.J5, a, b, winds, 3)
        for r, nw in ((3, 8), (2, 8), (8, 16), (1, 16)):
            assert l.shapes_rtile(C.byref(j), r, nw) != 0
        j.k = 16  # the halo of a 32-row tile
        assert l.shapes_rtile(C.byref(j), 2, 16) != 0


@pytest.mark.parametrize("r,nw", [(2, 8), (2, 16), (4, 8)])
def test_cloudsim_special_values(gpu, r, nw):
    """Infinities, NaN and huge values of the state and the winds reach the same cells
    (NaN wind compares as no wind: the lower neighbour is read)."""
    l = shapes.lib()
    a, b, (wx, wy), _ = _inputs(shapes.CLOUD, (75, 530))
    a[20, 255], a[40, 3], a[60, 256], a[33, 500], a[0, 7] = np.inf, np.nan, -np.inf, 3e38, np.inf
    wx[100, 30], wy[300, 50], wx[400, 10], wy[257, 41] = np.nan, np.inf, -np.inf, np.nan
    for k in (2, 5):
        with _Buffers() as bufs:
            j, am = _job(bufs, shapes.CLOUD, a, b, (wx, wy), k)
            assert l.shapes_rtile(C.byref(j), r, nw) == 0
            L.check(L.lib().pskel_device_synchronize())
            got = bufs.read(j.dst, am)[:, :a.shape[1]]
        np.testing.assert_array_equal(got, oracle.run_2d_cloud(a, wx, wy, 0.01, k, out=b))
