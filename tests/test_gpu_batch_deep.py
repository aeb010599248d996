"""Batches whose register-tile families fuse more sweeps per launch than asked:
runs long enough for the deepest tiles, then short ones of other lengths on the
same batch (each length has its own tiles), every grid equal to the oracle."""
import numpy as np
import pytest

import oracle
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu

SHAPES = [(3, 9, "jacobi2d"), (64, 256, "jacobi2d"), (65, 257, "diffusion9"), (333, 777, "jacobi2d"),
          (129, 1030, "diffusion9"), (64, 2048, "life"), (65, 2049, "life"), (500, 100, "life"), (2, 2, "life"),
          (40, 8, "jacobi2d")]  # the last: too narrow for the register tiles, LDS tiles of 3 sweeps


@pytest.mark.parametrize("use_graph", [True, False])
def test_batch_deep(gpu, use_graph):
    grids, stencils, fields, outs = [], [], [], []
    try:
        for i, (h, w, name) in enumerate(SHAPES):
            u = inputs.uniform(50 + i, 0, h * w).reshape(h, w)
            f = (u < np.float32(0.35)).astype(np.uint8) if name == "life" else u
            o = f.copy()  # another ring
            o[0, :], o[:, -1] = (1 - f[0, :], 1 - f[:, -1]) if name == "life" else (2.0, -1.0)
            g = api.Grid((h, w), "u8" if name == "life" else "f32")
            g.upload_pair(f, o)
            grids.append(g)
            stencils.append(getattr(K, name)())
            fields.append(f)
            outs.append(o)
        depths = [7 if s[2] == "life" else 3 for s in SHAPES]
        done = 0
        with api.Batch(grids, stencils, None, depths) as b:
            for n in (61, 1, 8, 61, 40):
                b.run(n, use_graph=use_graph)
                done += n
                for g, s, f, o in zip(grids, stencils, fields, outs):
                    assert np.array_equal(g.download(), oracle.run_2d(s, f, done, out=o)), (g.shape, n, done)
    finally:
        for g in grids:
            g.close()
