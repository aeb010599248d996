"""Both splits of the fused 3D march's planes over blocks against the CPU oracle,
bit-exact: grids with slightly more tiles than CUs (256) and few planes, whose
blocks take even ranges that end in one tile and go on in the next, and the same
grids one tile short of that, which take equal segments."""
import numpy as np
import pytest

import oracle
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile,block,depth,width", [((4, 4, 0), (512, 2), 3, 3100), ((4, 4, 0), (512, 2), 3, 3070),
                                                    ((4, 2, 0), (768, 2), 3, 2100), ((4, 2, 0), (768, 2), 3, 2040),
                                                    ((4, 3, 0), (768, 2), 2, 4100), ((4, 3, 0), (768, 2), 2, 4080)])
def test_fused_split(gpu, tile, block, depth, width):
    shape = (13, width, 20)
    a = inputs.uniform(width, 0, int(np.prod(shape))).reshape(shape)
    want, want_res = oracle.run_3d(K.jacobi3d(), a, 2 * depth, residual_every=depth)
    with api.Grid(shape, "f32") as g:
        g.upload_pair(a)
        st = g.run(K.jacobi3d(), 2 * depth, variant="tuned", tile=tile, block=block, time_tile=depth,
                   residual_every=depth)
        got = g.download()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    np.testing.assert_allclose(st["residuals"], want_res, rtol=1e-12, atol=0)
