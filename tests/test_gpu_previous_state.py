"""download_previous and grid_residual after 2D runs whose launches are deeper than
the depth they name: where launches of that depth end in a single sweep (on a
residual step, with one sweep left over, and always for CLOUDSIM), the other buffer
holds the state one sweep before the result, bit-equal to the oracle's, its own
ring included.  The residual is an FP64 sum over the same cells in another order:
within 1e-12."""
import numpy as np
import pytest

import oracle
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu

# sweeps, time_tile, residual_every
RUNS = [(9, 4, 0), (16, 3, 0), (20, 4, 20), (21, 2, 7), (10, 4, 5), (41, 4, 40), (1, 4, 0)]
CLOUD_RUNS = [(8, 4, 0), (11, 2, 0), (2, 4, 0), (20, 4, 20), (23, 4, 7)]


def _case(name, shape):
    n = shape[0] * shape[1]
    if name == "cloudsim":
        a, wx, wy = inputs.cloudsim_fields(*shape, seed=sum(shape))
    else:
        a, wx, wy = inputs.uniform(sum(shape), 0, n).reshape(shape), None, None
    if name == "life":
        a = (a < np.float32(0.35)).astype(np.uint8)
    b = a.copy()  # another ring
    if name == "life":
        b[0, :], b[:, -1] = 1 - a[0, :], 1 - a[:, -1]
    else:
        b[0, :], b[-1, :], b[:, 0], b[:, -1] = 3.0, -2.0, 0.5, 7.0
    s = K.cloudsim(0.01) if name == "cloudsim" else getattr(K, name)()

    def state(k):
        if k == 0:
            return a
        return oracle.run_2d_cloud(a, wx, wy, 0.01, k, out=b) if name == "cloudsim" else oracle.run_2d(s, a, k, out=b)

    return s, a, b, wx, wy, state


@pytest.mark.parametrize("use_graph", [False, True])
@pytest.mark.parametrize("shape", [(33, 257), (130, 94), (400, 1303)])
@pytest.mark.parametrize("name", ["jacobi2d", "diffusion9", "cloudsim", "life"])
def test_previous_state(gpu, name, shape, use_graph):
    s, a, b, wx, wy, state = _case(name, shape)
    fields = [api.Field(wx), api.Field(wy)] if name == "cloudsim" else []
    try:
        for n, k, every in CLOUD_RUNS if name == "cloudsim" else RUNS:
            with api.Grid(shape, "u8" if name == "life" else "f32") as g:
                for i, f in enumerate(fields):
                    g.set_field(i, f)
                for rep in range(2 if use_graph else 1):
                    g.upload_pair(a, b)
                    g.run(s, n, variant="tuned", time_tile=k, residual_every=every, use_graph=use_graph)
                    got, prev, r = g.download(), g.download_previous(), g.residual()
                    want, before = state(n), state(n - 1)
                    assert np.array_equal(got.view(np.uint8), want.view(np.uint8)), (n, k, every, rep)
                    assert np.array_equal(prev.view(np.uint8), before.view(np.uint8)), (n, k, every, rep)
                    d = np.linalg.norm(want.astype(np.float64) - before.astype(np.float64))
                    np.testing.assert_allclose(r, d, rtol=1e-12, atol=0)
                # the next run reads both buffers
                g.run(s, 7, variant="tuned", time_tile=4)
                assert np.array_equal(g.download().view(np.uint8), state(n + 7).view(np.uint8)), (n, k, every)
    finally:
        for f in fields:
            f.close()
