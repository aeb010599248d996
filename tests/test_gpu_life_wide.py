"""Boards too wide for the bit-packed tiles (8M columns) run one generation per launch,
whatever fused tile the launch names."""
import numpy as np
import pytest

import oracle
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [0, 24, 48])
def test_wide_board(gpu, rows):
    h, w = 5, (1 << 23) + 77
    a = (inputs.uniform(31, 0, h * w).reshape(h, w) < np.float32(0.35)).astype(np.uint8)
    with api.Grid((h, w), "u8") as g:
        g.upload_pair(a)
        st = g.run(K.life(), 5, variant="tuned", time_tile=8, tile=(0, rows, 0), residual_every=3)
        assert st["launches"] == 5
        assert np.array_equal(g.download(), oracle.run_2d(K.life(), a, 5))
