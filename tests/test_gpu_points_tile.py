"""The LDS tile of arbitrary masks, launched directly (a run takes it only where it is
faster than the plain kernel): one sweep, bit-equal to the oracle, on grids at the
tiles' edges and thin in each axis, with partials (FP64 sums over the same cells in
another order: within 1e-12)."""
import ctypes as C

import numpy as np
import pytest

import oracle
import shapes
from pskel_amd import _lib as L
from pskel_amd import inputs
from pskel_amd import kernels as K
from test_gpu_points import MASKS, SHAPES, _mask
from test_gpu_tile_shapes import _Buffers, _same

pytestmark = pytest.mark.gpu

THIN = [(1, 300, 70), (70, 1, 300), (300, 70, 1), (2, 3, 900)]


def _pitched(a):
    rows = a.reshape(-1, a.shape[-1])
    pitch = -(-rows.shape[1] * a.itemsize // 1024) * 1024 // a.itemsize
    m = np.zeros((rows.shape[0], pitch), a.dtype)
    m[:, :rows.shape[1]] = rows
    return m


@pytest.mark.parametrize("mask", list(MASKS))
@pytest.mark.parametrize("kind", [K.SCALED_SUM, K.WEIGHTED_SUM])
@pytest.mark.parametrize("boundary", [K.BOUNDARY_COPY, K.BOUNDARY_HALO])
def test_tile_3d(gpu, mask, kind, boundary):
    l = shapes.lib()
    for shape in SHAPES + THIN:
        s = _mask(mask, kind, 3, boundary=boundary, halo_value=0.75)
        d = s.desc()
        a = inputs.uniform(sum(shape), 0, int(np.prod(shape))).reshape(shape)
        want, _ = oracle.run_3d(s, a, 1)
        h, w, dd = shape
        nb = l.shapes_points_blocks(C.byref(d), w, h, dd)
        assert nb > 0
        m, part = _pitched(a), np.full(nb, np.nan)
        for residual in (False, True):
            with _Buffers() as bufs:
                src, dst, pp = bufs.new(m), bufs.new(np.zeros_like(m)), bufs.new(part)
                assert l.shapes_points(C.addressof(d), 3, src, dst, pp if residual else None, w, h, dd, m.shape[1],
                                       L.DTYPE_F32, 0.0, L.ROUND_NEAREST, 0, 0) == 0, shape
                L.check(L.lib().pskel_device_synchronize())
                _same(bufs.read(dst, m), want.reshape(-1, dd), (shape, residual))
                if residual:
                    diff = want.astype(np.float64) - a.astype(np.float64)
                    np.testing.assert_allclose(bufs.read(pp, part).sum(), (diff * diff).sum(), rtol=1e-12, atol=0)


@pytest.mark.parametrize("store", ["bf16", "f16"])
@pytest.mark.parametrize("rounding", ["nearest", "stochastic"])
@pytest.mark.parametrize("kind", [K.SCALED_SUM, K.WEIGHTED_SUM])
@pytest.mark.parametrize("boundary", [K.BOUNDARY_COPY, K.BOUNDARY_HALO])
def test_tile_3d_16bit(gpu, store, rounding, kind, boundary):
    l = shapes.lib()
    code = oracle.STORE_BF16 if store == "bf16" else oracle.STORE_F16
    rc = oracle.ROUND_STOCHASTIC if rounding == "stochastic" else oracle.ROUND_NEAREST
    for shape in ((9, 17, 65), (5, 30, 131), (2, 3, 900)):
        s = _mask("box27", kind, 3, boundary=boundary, halo_value=0.75)
        d = s.desc()
        words = (inputs.uniform(3, 0, int(np.prod(shape))) * np.float32(2.0)).view(np.uint32).reshape(shape)
        words = (words >> 16).astype(np.uint16) & np.uint16(0xBFFF)  # finite in either format
        want = oracle.run_3d_r16(s, code, words, 1, store_offset=0.5, rounding=rc, seed=5)[0]
        h, w, dd = shape
        m = _pitched(words)
        with _Buffers() as bufs:
            src, dst = bufs.new(m), bufs.new(np.zeros_like(m))
            assert l.shapes_points(C.addressof(d), 3, src, dst, None, w, h, dd, m.shape[1],
                                   {"bf16": L.DTYPE_BF16, "f16": L.DTYPE_F16}[store], 0.5,
                                   {"nearest": L.ROUND_NEAREST, "stochastic": L.ROUND_STOCHASTIC}[rounding], 5, 0) == 0
            L.check(L.lib().pskel_device_synchronize())
            _same(bufs.read(dst, m), want.reshape(-1, dd), shape)


@pytest.mark.parametrize("mask", list(MASKS))
@pytest.mark.parametrize("kind", [K.SCALED_SUM, K.WEIGHTED_SUM])
def test_tile_2d(gpu, mask, kind):
    l = shapes.lib()
    for shape in ((1, 1), (65, 130), (64, 64), (129, 33), (257, 17), (3, 700), (700, 3)):
        s = _mask(mask, kind, 2)
        d = s.desc()
        a = inputs.jacobi2d_field(*shape, seed=sum(shape))
        b = np.full_like(a, 2.0)  # its ring is kept
        want = oracle.run_2d(s, a, 1, out=b)
        m = _pitched(a)
        with _Buffers() as bufs:
            src, dst = bufs.new(m), bufs.new(_pitched(b))
            assert l.shapes_points(C.addressof(d), 2, src, dst, None, shape[1], shape[0], 1, m.shape[1], L.DTYPE_F32,
                                   0.0, L.ROUND_NEAREST, 0, 0) == 0
            L.check(L.lib().pskel_device_synchronize())
            _same(bufs.read(dst, m), want, shape)
