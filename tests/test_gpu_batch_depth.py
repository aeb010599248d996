"""The depth of a batch's tile families: at least what each grid asks for.  The work
items show it: tall boards need more tiles the deeper the launch, so a batch in
which one board asks for 7 generations has the tiles of one in which all do."""
import numpy as np
import pytest

import oracle
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu

SHAPES = [(1500, 200), (1500, 300), (1500, 100)]


def _items(depths, n):
    """the batch's items after a run of n generations (checked against the oracle)"""
    boards = [(inputs.uniform(90 + i, 0, h * w).reshape(h, w) < np.float32(0.35)).astype(np.uint8)
              for i, (h, w) in enumerate(SHAPES)]
    grids = [api.Grid(b.shape, "u8") for b in boards]
    try:
        for g, b in zip(grids, boards):
            g.upload_pair(b)
        with api.Batch(grids, [K.life()] * len(grids), None, depths) as batch:
            batch.run(n)
            for g, b in zip(grids, boards):
                assert np.array_equal(g.download(), oracle.run_2d(K.life(), b, n)), (depths, g.shape)
            return batch.info()["items"]
    finally:
        for g in grids:
            g.close()


def test_deepest_ask_holds(gpu):
    # 6 generations are two launches at depth 3, 5 and 7: the shallowest has the fewest tiles
    assert _items([3, 3, 3], 6) < _items([7, 7, 7], 6)
    for depths in ([3, 7, 3], [7, 3, 5], [3, 3, 7]):
        assert _items(depths, 6) == _items([7, 7, 7], 6), depths
