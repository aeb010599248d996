"""GPU parity of the 2D register tiles (fused sweeps of the 5-point, 9-point and
CLOUDSIM stencils) against the CPU oracle, bit-exact: both sides round every
product and sum on its own in the same order.  Grids sit at the tiles' edges
(256 columns, 16 to 64 rows), runs at the ends of the depths (one sweep, odd and
even, longer than the deepest launch)."""
import numpy as np
import pytest

import oracle
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu

SHAPES = [(3, 9), (16, 255), (32, 256), (33, 257), (64, 10), (65, 497), (130, 94), (200, 1300), (700, 700), (31, 4000)]
RUNS = (1, 2, 7, 16, 33, 71)


def _rings(a):
    """a distinct output ring: every fused sweep reads the ring of its own buffer"""
    b = a.copy()
    b[0, :], b[-1, :], b[:, 0], b[:, -1] = 3.0, -2.0, 0.5, 7.0
    return b


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("name", ["jacobi2d", "diffusion9"])
def test_rtile_parity(gpu, shape, name):
    s = getattr(K, name)()
    a = inputs.uniform(sum(shape), 0, shape[0] * shape[1]).reshape(shape)
    b = _rings(a)
    for n in RUNS:
        want = oracle.run_2d(s, a, n, out=b)
        with api.Grid(shape, "f32") as g:
            g.upload_pair(a, b)
            g.run(s, n, variant="tuned", time_tile=4)
            assert np.array_equal(g.download().view(np.uint32), want.view(np.uint32)), (shape, n)


@pytest.mark.parametrize("shape", SHAPES)
def test_rtile_cloudsim(gpu, shape):
    t, wx, wy = inputs.cloudsim_fields(*shape, seed=sum(shape))
    wx[0, :3] = (0.0, -0.0, 0.5)  # no wind reads the lower neighbour
    s = K.cloudsim(0.01)
    with api.Field(wx) as fx, api.Field(wy) as fy:
        for n in RUNS:
            want = oracle.run_2d_cloud(t, wx, wy, 0.01, n)
            with api.Grid(shape, "f32") as g:
                g.set_field(0, fx)
                g.set_field(1, fy)
                g.upload_pair(t)
                g.run(s, n, variant="tuned", time_tile=4)
                assert np.array_equal(g.download().view(np.uint32), want.view(np.uint32)), (shape, n)


@pytest.mark.parametrize("name", ["jacobi2d", "diffusion9"])
def test_rtile_special_values(gpu, name):
    """Infinities, NaN and huge values reach the same cells."""
    s = getattr(K, name)()
    a = inputs.uniform(5, 0, 130 * 300).reshape(130, 300)
    a[40, 255], a[64, 0], a[100, 256], a[129, 299], a[7, 7] = np.inf, np.nan, -np.inf, np.inf, 3e38
    with api.Grid(a.shape, "f32") as g:
        g.upload_pair(a)
        g.run(s, 20, variant="tuned", time_tile=4)
        np.testing.assert_array_equal(g.download(), oracle.run_2d(s, a, 20))


@pytest.mark.parametrize("every", [1, 6, 20])
def test_rtile_residuals_resume_and_graph(gpu, every):
    """Residuals reduced inside the single sweep that ends an interval, runs that
    resume, and three replays of one captured graph."""
    s = K.diffusion9()
    a = inputs.uniform(6, 0, 300 * 519).reshape(300, 519)
    b = _rings(a)
    states = [oracle.run_2d(s, a, n, out=b) for n in range(0, 61)]
    want = [np.linalg.norm(states[n].astype(np.float64) - states[n - 1].astype(np.float64)) for n in range(1, 61)]
    # the first sweep's state before it is `a`, whose ring its own buffer keeps
    want[0] = np.linalg.norm(states[1].astype(np.float64) - a.astype(np.float64))
    with api.Grid(a.shape, "f32") as g:
        g.upload_pair(a, b)
        for rep in range(3):
            st = g.run(s, 20, variant="tuned", time_tile=4, residual_every=every, use_graph=True)
            api.synchronize()
            done = 20 * (rep + 1)
            assert np.array_equal(g.download().view(np.uint32), states[done].view(np.uint32)), rep
            exp = [want[n - 1] for n in range(done - 20 + 1, done + 1) if (n - (done - 20)) % every == 0]
            np.testing.assert_allclose(st["residuals"], exp, rtol=1e-12, atol=0)
