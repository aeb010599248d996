"""The other buffer of batched grids: where launches of the depth asked for end in a
single sweep, it holds the state one sweep before the result, at whatever depth the
batch runs, bit-equal to the oracle's, ring included."""
import numpy as np
import pytest

import oracle
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu

# (h, w, stencil, depth asked)
GRIDS = [(65, 257, "jacobi2d", 3), (130, 94, "diffusion9", 3), (70, 300, "life", 3), (33, 64, "life", 5),
         (200, 2049, "life", 7), (20, 30, "jacobi2d", 1)]


def _ends_single(n, k):
    r = n % k
    return k == 1 or r == 1 or (r > 0 and r % 2 == 0)


@pytest.mark.parametrize("use_graph", [True, False])
def test_batch_previous_state(gpu, use_graph):
    grids, stencils, fields, outs = [], [], [], []
    try:
        for i, (h, w, name, _) in enumerate(GRIDS):
            u = inputs.uniform(80 + i, 0, h * w).reshape(h, w)
            f = (u < np.float32(0.35)).astype(np.uint8) if name == "life" else u
            o = f.copy()  # another ring
            o[0, :], o[:, -1] = (1 - f[0, :], 1 - f[:, -1]) if name == "life" else (2.0, -1.0)
            g = api.Grid((h, w), "u8" if name == "life" else "f32")
            grids.append(g)
            stencils.append(getattr(K, name)())
            fields.append(f)
            outs.append(o)
        seen = 0
        with api.Batch(grids, stencils, None, [k for *_, k in GRIDS]) as b:
            for n in (5, 8, 11, 20, 34, 104, 1, 2):
                for g, f, o in zip(grids, fields, outs):
                    g.upload_pair(f, o)
                b.run(n, use_graph=use_graph)
                for g, s, f, o, (h, w, name, k) in zip(grids, stencils, fields, outs, GRIDS):
                    assert np.array_equal(g.download(), oracle.run_2d(s, f, n, out=o)), (name, h, n)
                    if _ends_single(n, k):
                        before = oracle.run_2d(s, f, n - 1, out=o) if n > 1 else f
                        assert np.array_equal(g.download_previous(), before), (name, h, n)
                        seen += 1
        assert seen > 20
    finally:
        for g in grids:
            g.close()
