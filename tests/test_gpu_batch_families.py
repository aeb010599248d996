"""Batches of f32 grids that name LDS tiles take those where they are faster (few or
narrow 3x3 grids, short runs of both stencils together), else register tiles; both
again for other run lengths on the same batch.  The launches show which (the LDS tiles
run 3 sweeps a launch); every grid equals the oracle."""
import numpy as np
import pytest

import oracle
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu

SMALL = [(70, 300, "diffusion9"), (129, 600, "diffusion9")]
NARROW = [(4000, 60, "diffusion9"), (900, 100, "diffusion9")] * 4
WIDE = [(700, 700, "diffusion9")] * 6
MIXED = [(300, 500, "jacobi2d"), (200, 400, "diffusion9")]
FIVE = [(300, 500, "jacobi2d"), (90, 260, "jacobi2d")]


@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("shapes,lds", [(SMALL, [30, 60]), (NARROW, [30, 60]), (WIDE, []), (MIXED, [9, 30]), (FIVE, [])])
def test_families(gpu, shapes, lds, use_graph):
    grids, stencils, fields, outs = [], [], [], []
    try:
        for i, (h, w, name) in enumerate(shapes):
            f = inputs.uniform(60 + i, 0, h * w).reshape(h, w)
            o = f.copy()
            o[0, :], o[:, -1] = 2.0, -1.0
            grids.append(api.Grid((h, w), "f32"))
            stencils.append(getattr(K, name)())
            fields.append(f)
            outs.append(o)
        with api.Batch(grids, stencils, None, [3] * len(grids)) as b:
            for n in (9, 30, 1, 60, 9):
                for g, f, o in zip(grids, fields, outs):
                    g.upload_pair(f, o)
                launches = b.run(n, use_graph=use_graph)["launches"]
                if n in lds:
                    assert launches == n // 3, n
                elif n >= 30 and not lds:
                    assert launches < n // 3, n
                for g, s, f, o in zip(grids, stencils, fields, outs):
                    assert np.array_equal(g.download(), oracle.run_2d(s, f, n, out=o)), (g.shape, n)
    finally:
        for g in grids:
            g.close()
