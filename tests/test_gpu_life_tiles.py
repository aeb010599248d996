"""Bit-packed life tiles (many generations per launch) against the CPU oracle,
bit-exact: boards at the edges of the tiles (lanes of 32 columns, 2048 columns,
16 to 128 rows), generations odd and even and beyond the deepest launch, distinct
rings, resumed runs and graph replays."""
import numpy as np
import pytest

import oracle
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (3, 3), (5, 33), (16, 32), (17, 64), (32, 2047), (33, 2048), (65, 2049), (129, 2081), (300, 97),
          (1000, 1503), (40, 6100), (700, 31)]


def _board(shape, seed):
    return (inputs.uniform(seed, 0, shape[0] * shape[1]).reshape(shape) < np.float32(0.35)).astype(np.uint8)


@pytest.mark.parametrize("shape", SHAPES)
def test_life_tiles(gpu, shape):
    a = _board(shape, sum(shape))
    b = a.copy()  # another ring: alive where the input's is dead
    b[0, :], b[-1, :], b[:, 0], b[:, -1] = 1 - a[0, :], 1 - a[-1, :], 1 - a[:, 0], 1 - a[:, -1]
    for n in (1, 2, 7, 16, 31, 77):
        with api.Grid(shape, "u8") as g:
            g.upload_pair(a, b)
            g.run(K.life(), n, variant="tuned", time_tile=8)
            assert np.array_equal(g.download(), oracle.run_2d(K.life(), a, n, out=b)), (shape, n)


def test_life_tiles_resume_graph_residual(gpu):
    a = _board((331, 2100), 9)
    with api.Grid(a.shape, "u8") as g:
        g.upload_pair(a)
        for rep in range(1, 4):
            st = g.run(K.life(), 25, variant="tuned", time_tile=7, residual_every=25, use_graph=True)
            api.synchronize()
            want = oracle.run_2d(K.life(), a, 25 * rep)
            prev = oracle.run_2d(K.life(), a, 25 * rep - 1)
            assert np.array_equal(g.download(), want), rep
            assert st["residuals"] == [float(np.linalg.norm(want.astype(np.float64) - prev))], rep
