"""3D grids less than four cells wide: the launch chosen for an arbitrary mask spreads its
block along the depth, and computes what any other block does."""
import itertools

import numpy as np
import pytest

from pskel_amd import api, inputs, tuner
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,block", [((37, 1, 256), (256, 1)), ((37, 2, 300), (128, 2)), ((40, 3, 257), (256, 1)),
                                         ((37, 2, 255), (0, 0)), ((37, 4, 300), (0, 0))])
@pytest.mark.parametrize("boundary", [0, 1])
@pytest.mark.parametrize("storage", ["f32", "bf16"])
def test_chosen_block(gpu, shape, block, boundary, storage):
    mask = list(itertools.product((-1, 0, 1), repeat=3))
    s = K.Stencil(K.WEIGHTED_SUM, 3, mask, weights=[1.0 / 27] * 27, boundary=boundary, halo_value=0.5)
    cfg = tuner.choose_config(s, shape, storage, 5)
    assert cfg["variant"] == "tuned" and tuple(cfg["block"]) == block
    a = inputs.uniform(9, 0, int(np.prod(shape))).reshape(shape)
    got = []
    for kw in (cfg, {"variant": "plain", "block": (64, 1)}):
        with api.Grid(shape, storage) as g:
            g.upload_pair(a)
            g.run(s, 5, **kw)
            got.append(g.download())
    assert np.array_equal(got[0], got[1])
