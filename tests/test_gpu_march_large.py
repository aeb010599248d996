"""The 9-point register march where runs still take it (grids above 12M cells): odd
width, distinct rings, depths 2 to 4 as run tails and before residual steps, bit-equal
to the oracle.  Residuals are FP64 sums in another order: within 1e-12."""
import numpy as np
import pytest

import oracle
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu

SHAPE = (2801, 4399)


@pytest.fixture(scope="module")
def case():
    a = inputs.uniform(17, 0, SHAPE[0] * SHAPE[1]).reshape(SHAPE)
    b = a.copy()
    b[0, :], b[-1, :], b[:, 0], b[:, -1] = 3.0, -2.0, 0.5, 7.0
    s = K.diffusion9()
    states = {0: a}
    for n in (4, 5, 7, 8, 9, 10):
        states[n] = oracle.run_2d(s, a, n, out=b)
    return s, a, b, states


@pytest.mark.parametrize("tile", [(4, 0, 0), (4, 0, 24), (4, 0, 7), (0, 32, 0)])
@pytest.mark.parametrize("n,k", [(9, 4), (8, 3), (10, 4), (7, 2)])
def test_large_march(gpu, case, tile, n, k):
    s, a, b, states = case
    with api.Grid(SHAPE, "f32") as g:
        g.upload_pair(a, b)
        st = g.run(s, n, variant="tuned", time_tile=k, tile=tile)
        assert st["launches"] == -(-n // k)  # launches of the depth named, not the register tiles'
        assert np.array_equal(g.download().view(np.uint32), states[n].view(np.uint32))


@pytest.mark.parametrize("use_graph", [False, True])
def test_large_march_residuals(gpu, case, use_graph):
    s, a, b, states = case
    want = [np.linalg.norm(states[n].astype(np.float64) - states[n - 1].astype(np.float64)) for n in (5, 10)]
    with api.Grid(SHAPE, "f32") as g:
        for rep in range(2):
            g.upload_pair(a, b)
            st = g.run(s, 10, variant="tuned", time_tile=4, tile=(4, 0, 0), residual_every=5, use_graph=use_graph)
            assert np.array_equal(g.download().view(np.uint32), states[10].view(np.uint32)), rep
            assert np.array_equal(g.download_previous().view(np.uint32), states[9].view(np.uint32)), rep
            np.testing.assert_allclose(st["residuals"], want, rtol=1e-12, atol=0)
