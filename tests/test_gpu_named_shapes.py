"""Launches that name a shape which is not built are refused where launches of the
depth they name would use it, whatever kernel runs instead; where single sweeps are
all they come to, they run.  The grid's state stays as it was after a refusal."""
import numpy as np
import pytest

import oracle
from pskel_amd import _lib as L
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu


def _grid(shape, seed=5):
    a = inputs.uniform(seed, 0, int(np.prod(shape))).reshape(shape)
    g = api.Grid(shape, "f32")
    g.upload_pair(a)
    return g, a


@pytest.mark.parametrize("name", ["jacobi2d", "diffusion9"])
def test_lds_tile_rows(gpu, name):
    s = getattr(K, name)()
    g, a = _grid((90, 300))
    with g:
        for rows in (1, 13, 24, 128):
            for kw in ({}, {"residual_every": 3}, {"use_graph": True}):
                with pytest.raises(L.PSkelError):
                    g.run(s, 9, variant="tuned", time_tile=4, tile=(0, rows, 0), **kw)
        assert np.array_equal(g.download(), a)
        # single sweeps throughout: a run of one, a residual every sweep or two
        g.run(s, 1, variant="tuned", time_tile=4, tile=(0, 13, 0))
        g.run(s, 4, variant="tuned", time_tile=4, tile=(0, 13, 0), residual_every=1)
        g.run(s, 4, variant="tuned", time_tile=4, tile=(0, 13, 0), residual_every=2)
        for rows in (-1, 0, 8, 16, 32, 64):
            g.run(s, 9, variant="tuned", time_tile=4, tile=(0, rows, 0))
        assert np.array_equal(g.download(), oracle.run_2d(s, a, 63))


def test_cloudsim_rows_and_waves(gpu):
    t, wx, wy = inputs.cloudsim_fields(70, 200, seed=9)
    s = K.cloudsim(0.01)
    with api.Grid(t.shape, "f32") as g, api.Field(wx) as fx, api.Field(wy) as fy:
        g.set_field(0, fx)
        g.set_field(1, fy)
        g.upload_pair(t)
        for tile in ((0, 3, 0), (0, 16, 0), (0, 2, 5)):
            with pytest.raises(L.PSkelError):
                g.run(s, 6, variant="tuned", time_tile=4, tile=tile)
        for tile in ((0, 0, 0), (0, 8, 4), (7, 1, 1)):
            g.run(s, 6, variant="tuned", time_tile=4, tile=tile)
        assert np.array_equal(g.download(), oracle.run_2d_cloud(t, wx, wy, 0.01, 18))


def test_block_of_an_arbitrary_mask(gpu):
    s = K.Stencil(K.WEIGHTED_SUM, 3, [(0, 0, 0), (1, 0, 0), (0, 0, 1)], weights=[0.5, 0.25, 0.25])
    g, a = _grid((64, 64, 80))  # large enough for the LDS tile of any mask
    with g:
        for block in ((64, 32), (2048, 1)):
            with pytest.raises(L.PSkelError):
                g.run(s, 2, variant="tuned", block=block)
        assert np.array_equal(g.download(), a)
        g.run(s, 2, variant="tuned", block=(64, 16))
        assert np.array_equal(g.download(), oracle.run_3d(s, a, 2)[0])
