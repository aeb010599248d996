"""CLOUDSIM with wind fields of different extents (each at least the grid's): each
field has its own row pitch on the device.  Bit-equal to the oracle on the fields'
common part, on every kernel, in either slot."""
import numpy as np
import pytest

import oracle
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [{"variant": "plain"}, {"variant": "tuned"}, {"variant": "tuned", "time_tile": 4},
                                {"variant": "tuned", "time_tile": 4, "residual_every": 5}])
@pytest.mark.parametrize("wide", [0, 1])
def test_cloud_fields_of_different_extents(gpu, wide, kw):
    h, w = 70, 200
    t, wx, wy = inputs.cloudsim_fields(h, w, seed=8)
    want = oracle.run_2d_cloud(t, wx, wy, 0.01, 10)
    fields = [wx, wy]
    # rows of 768 cells where the other field has 256, and more rows than the grid
    big = np.full((600, h + 30), -9.0, np.float32)
    big[:w, :h] = fields[wide]
    fields[wide] = big
    with api.Grid((h, w), "f32") as g, api.Field(fields[0]) as fx, api.Field(fields[1]) as fy:
        g.set_field(0, fx)
        g.set_field(1, fy)
        g.upload_pair(t)
        g.run(K.cloudsim(0.01), 10, **kw)
        assert np.array_equal(g.download().view(np.uint32), want.view(np.uint32))
