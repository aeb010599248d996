"""Residuals reduced inside the register-tile launch that ends an interval, however
many sweeps it fuses: ||u^n - u^(n-1)||, ring cells included, against the CPU
oracle's states.  Both sums are FP64 over the same bit-exact cells, in another
order: they agree to a few times the cell count's rounding, 1e-12 here."""
import numpy as np
import pytest

import oracle
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["jacobi2d", "diffusion9", "cloudsim"])
@pytest.mark.parametrize("shape", [(3, 9), (33, 257), (130, 94), (65, 497), (400, 1300)])
@pytest.mark.parametrize("every", [2, 3, 7, 16, 45])
def test_rtile_fused_residual(gpu, name, shape, every):
    n = 2 * every + 1
    if name == "cloudsim":
        s = K.cloudsim(0.01)
        a, wx, wy = inputs.cloudsim_fields(*shape, seed=sum(shape))
    else:
        s = getattr(K, name)()
        a = inputs.uniform(sum(shape), 0, shape[0] * shape[1]).reshape(shape)
    b = a.copy()  # a distinct ring: it changes with every sweep
    b[0, :], b[-1, :], b[:, 0], b[:, -1] = 3.0, -2.0, 0.5, 7.0

    def state(k):
        if name == "cloudsim":
            return oracle.run_2d_cloud(a, wx, wy, 0.01, k, out=b)
        return oracle.run_2d(s, a, k, out=b)

    want = [np.linalg.norm(state(k).astype(np.float64) - state(k - 1).astype(np.float64)) for k in (every, 2 * every)]
    with api.Grid(shape, "f32") as g:
        fields = [api.Field(wx), api.Field(wy)] if name == "cloudsim" else []
        for i, f in enumerate(fields):
            g.set_field(i, f)
        g.upload_pair(a, b)
        st = g.run(s, n, variant="tuned", time_tile=4, residual_every=every)
        got = g.download()
        for f in fields:
            f.close()
    assert np.array_equal(got.view(np.uint32), state(n).view(np.uint32))
    np.testing.assert_allclose(st["residuals"], want, rtol=1e-12, atol=0)


def test_rtile_residual_beyond_the_depth(gpu):
    """An interval longer than several launches of the deepest kind."""
    s = K.jacobi2d()
    a = inputs.uniform(4, 0, 130 * 300).reshape(130, 300)
    want = np.linalg.norm(oracle.run_2d(s, a, 150).astype(np.float64) - oracle.run_2d(s, a, 149).astype(np.float64))
    with api.Grid(a.shape, "f32") as g:
        g.upload_pair(a)
        st = g.run(s, 160, variant="tuned", time_tile=4, residual_every=150)
    np.testing.assert_allclose(st["residuals"], [want], rtol=1e-12, atol=0)
