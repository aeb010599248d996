"""The single generations of a fused launch (residual steps, a last one left over) run on
tiles of their own, by the board's size: odd boards on both sides of that line, tall ones
whose tiles outnumber 65536, and last rows that fill a tile in part."""
import numpy as np
import pytest

import oracle
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1), (3, 5), (9, 1025), (203, 197), (1733, 1731), (1731, 1735), (20001, 157),
                                   (1200003, 2), (1500005, 3)])
def test_single_generations(gpu, shape):
    a = (inputs.uniform(37, 0, shape[0] * shape[1]).reshape(shape) < np.float32(0.35)).astype(np.uint8)
    with api.Grid(shape, "u8") as g:
        g.upload_pair(a)
        st = g.run(K.life(), 4, variant="tuned", time_tile=8, tile=(0, 24, 0), residual_every=1)
        assert st["launches"] == 4
        states = [oracle.run_2d(K.life(), a, n) for n in range(5)]
        assert np.array_equal(g.download(), states[4])
        assert st["residuals"] == [float(np.sqrt((p != q).sum())) for p, q in zip(states, states[1:])]
