"""Tall 9-point grids that one column of LDS tiles covers, with residuals eight sweeps or
more apart, take the LDS tiles their launches name (up to 1.5 times as fast there); closer
residuals, shorter or wider grids the register tiles, which reduce in their own launch."""
import numpy as np
import pytest

import oracle
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu


def _run(shape, n, every, tile):
    a, s = inputs.uniform(6, 0, shape[0] * shape[1]).reshape(shape), K.diffusion9()
    with api.Grid(shape, "f32") as g:
        g.upload_pair(a)
        st = g.run(s, n, variant="tuned", time_tile=4, tile=tile, residual_every=every)
        assert np.array_equal(g.download().view(np.uint32), oracle.run_2d(s, a, n).view(np.uint32))
    want = [np.linalg.norm(oracle.run_2d(s, a, m).astype(np.float64) - oracle.run_2d(s, a, m - 1))
            for m in range(every, n + 1, every)]
    np.testing.assert_allclose(st["residuals"], want, rtol=1e-12)
    return st["launches"]


@pytest.mark.parametrize("shape,every,tile,launches", [
    ((11201, 60), 8, (0, 16, 0), 6),     # 4 + 3 + 1 sweeps an interval
    ((9001, 60), 8, (0, 8, 0), 6),
    ((11201, 3), 9, (0, 8, 0), 6),       # 4 + 4 + 1
    ((13601, 120), 12, (0, 16, 0), 8),   # 4 + 4 + 3 + 1
    ((22401, 20), 8, (0, 32, 0), 6),
    ((22401, 20), 8, (0, 0, 0), 6),
])
def test_lds_tiles(gpu, shape, every, tile, launches):
    assert _run(shape, 2 * every, every, tile) == launches


@pytest.mark.parametrize("shape,every,tile", [
    ((9000, 60), 8, (0, 8, 0)),
    ((11200, 60), 8, (0, 16, 0)),
    ((13600, 61), 8, (0, 16, 0)),
    ((22400, 20), 8, (0, 32, 0)),
    ((13601, 121), 8, (0, 16, 0)),
    ((11201, 60), 7, (0, 16, 0)),
    ((11201, 60), 8, (4, 0, 0)),
])
def test_register_tiles(gpu, shape, every, tile):
    assert _run(shape, 2 * every, every, tile) < 6
