"""GPU parity of the LDS tile of arbitrary masks (the tuned variant's kernel for
stencils without a specialised one) against the CPU oracle, bit-exact: the sums
run in mask order on both sides.  Sizes sit at the tile's edges (8 planes x 8
rows x 64 cells, 16 x 8 x 32, 32 x 8 x 16; 2D 64 x 64, 128 x 32, 256 x 16)."""
import numpy as np
import pytest

import oracle
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu

BOX27 = [(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)]
STAR13 = [(0, 0, 0)] + [tuple(s * k if i == j else 0 for j in range(3)) for k in (1, 2) for i in range(3) for s in (-1, 1)]
SKEW = [(2, -1, 5), (0, 0, -3), (-1, 1, 0), (0, -2, 8)]       # lopsided reach, two halo granules along d
ONE = [(0, 1, 0)]
MASKS = {"box27": BOX27, "star13": STAR13, "skew": SKEW, "one": ONE}
# grids of 256K cells and more, where short masks take the tile too, last
SHAPES = [(1, 1, 1), (8, 8, 64), (9, 17, 65), (17, 9, 33), (33, 7, 16), (5, 30, 131), (40, 11, 12), (65, 67, 66)]


def _mask(name, kind, ndim, **kw):
    offs = MASKS[name] if ndim == 3 else sorted({(o[0], o[2]) for o in MASKS[name]})
    w = [(0.3 + 0.1 * i) / len(offs) for i in range(len(offs))]
    return K.Stencil(kind, ndim, list(offs), weights=w, coeff=0.9 / len(offs), **kw)


@pytest.mark.parametrize("mask", list(MASKS))
@pytest.mark.parametrize("kind", [K.SCALED_SUM, K.WEIGHTED_SUM])
@pytest.mark.parametrize("boundary", [K.BOUNDARY_COPY, K.BOUNDARY_HALO])
def test_points_3d(gpu, mask, kind, boundary):
    for shape in SHAPES:
        s = _mask(mask, kind, 3, boundary=boundary, halo_value=0.75)
        a = inputs.uniform(sum(shape), 0, int(np.prod(shape))).reshape(shape)
        want, want_res = oracle.run_3d(s, a, 4, residual_every=2)
        with api.Grid(shape, "f32") as g:
            g.upload_pair(a)
            st = g.run(s, 4, variant="tuned", residual_every=2)
            got = g.download()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), shape
        np.testing.assert_allclose(st["residuals"], want_res, rtol=1e-12, atol=0)


@pytest.mark.parametrize("store", ["bf16", "f16"])
@pytest.mark.parametrize("rounding", ["nearest", "stochastic"])
@pytest.mark.parametrize("kind", [K.SCALED_SUM, K.WEIGHTED_SUM])
def test_points_3d_16bit(gpu, store, rounding, kind):
    """Storage words equal the oracle's 16-bit runner's, both roundings."""
    code = oracle.STORE_BF16 if store == "bf16" else oracle.STORE_F16
    rc = oracle.ROUND_STOCHASTIC if rounding == "stochastic" else oracle.ROUND_NEAREST
    for shape in ((9, 17, 65), (5, 30, 131)):
        s = _mask("box27", kind, 3, boundary=K.BOUNDARY_COPY)
        a = inputs.uniform(3, 0, int(np.prod(shape))).reshape(shape)
        with api.Grid(shape, store, store_offset=0.5, rounding=rounding, seed=5) as g:
            g.upload_pair(a)
            words = g.download(raw=True)
            g.run(s, 5, variant="tuned")
            got = g.download(raw=True)
        want = oracle.run_3d_r16(s, code, words, 5, store_offset=0.5, rounding=rc, seed=5)[0]
        assert np.array_equal(got, want), shape


@pytest.mark.parametrize("mask", list(MASKS))
@pytest.mark.parametrize("kind", [K.SCALED_SUM, K.WEIGHTED_SUM])
def test_points_2d(gpu, mask, kind):
    # the tile runs from 640K cells
    for shape in ((1, 1), (65, 130), (831, 801), (20011, 33), (40, 17003), (769, 897)):
        s = _mask(mask, kind, 2)
        a = inputs.jacobi2d_field(*shape, seed=sum(shape))
        b = a.copy()
        b[0, :] = 2.0  # distinct rings: neither is written
        with api.Grid(shape, "f32") as g:
            g.upload_pair(a, b)
            g.run(s, 5, variant="tuned")
            got = g.download()
        assert np.array_equal(got.view(np.uint32), oracle.run_2d(s, a, 5, out=b).view(np.uint32)), shape


def test_points_special_values(gpu):
    """Infinities and NaN reach the same cells, and a mask range above the reach
    widens the copied faces."""
    shape = (12, 13, 70)
    s = _mask("box27", K.WEIGHTED_SUM, 3, boundary=K.BOUNDARY_COPY)
    s.radius = 3
    a = inputs.uniform(9, 0, int(np.prod(shape))).reshape(shape)
    a[5, 6, 20], a[6, 6, 40], a[0, 0, 0] = np.inf, np.nan, -np.inf
    want, _ = oracle.run_3d(s, a, 3)
    with api.Grid(shape, "f32") as g:
        g.upload_pair(a)
        g.run(s, 3, variant="tuned")
        got = g.download()
    np.testing.assert_array_equal(got, want)


def test_points_halo_too_wide(gpu):
    """A mask whose halo does not fit the tile still runs (the plain kernel)."""
    offs = [(0, 0, -9), (0, 0, 0), (0, 0, 9)]
    s = K.Stencil(K.WEIGHTED_SUM, 3, offs, weights=[0.25, 0.5, 0.25], boundary=K.BOUNDARY_HALO, halo_value=1.0)
    a = inputs.uniform(2, 0, 6 * 7 * 80).reshape(6, 7, 80)
    want, _ = oracle.run_3d(s, a, 3)
    with api.Grid(a.shape, "f32") as g:
        g.upload_pair(a)
        g.run(s, 3, variant="tuned")
        got = g.download()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
