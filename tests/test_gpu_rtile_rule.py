"""Tall grids narrower than a register tile, and short runs on large ones, take the
kernels their launches name (which measured up to twice as fast there), others the
tiles: the launches of a run show which.  Bit-equal to the oracle either way."""
import numpy as np
import pytest

import oracle
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu


def _run(name, shape, n, **kw):
    h, w = shape
    if name == "cloudsim":
        a, wx, wy = inputs.cloudsim_fields(h, w, seed=3)
        s, want = K.cloudsim(0.01), oracle.run_2d_cloud(a, wx, wy, 0.01, n)
    else:
        a, s = inputs.uniform(4, 0, h * w).reshape(shape), getattr(K, name)()
        want = oracle.run_2d(s, a, n)
    with api.Grid(shape, "f32") as g:
        fields = [api.Field(wx), api.Field(wy)] if name == "cloudsim" else []
        for i, f in enumerate(fields):
            g.set_field(i, f)
        g.upload_pair(a)
        st = g.run(s, n, variant="tuned", time_tile=4, **kw)
        assert np.array_equal(g.download().view(np.uint32), want.view(np.uint32)), (name, shape, n)
        for f in fields:
            f.close()
    return st["launches"]


@pytest.mark.parametrize("name,shape,n,kw,launches", [
    ("diffusion9", (9000, 40), 40, {"tile": (0, 16, 0)}, 10),
    ("diffusion9", (14000, 120), 21, {"tile": (0, 32, 0)}, 6),
    ("diffusion9", (2000, 2000), 3, {"tile": (4, 0, 0)}, 1),
    ("diffusion9", (20001, 50), 2, {"tile": (4, 0, 8)}, 1),
    ("jacobi2d", (7000, 60), 3, {"tile": (0, 16, 0)}, 1),
    ("cloudsim", (9000, 100), 3, {}, 3),
    ("cloudsim", (26000, 40), 7, {}, 7),
])
def test_named_kernels(gpu, name, shape, n, kw, launches):
    assert _run(name, shape, n, **kw) == launches


@pytest.mark.parametrize("name,shape,n,kw", [
    ("diffusion9", (1500, 40), 40, {"tile": (0, 16, 0)}),
    ("diffusion9", (9000, 40), 40, {"tile": (0, 16, 0), "residual_every": 20}),
    ("diffusion9", (9000, 121), 40, {"tile": (0, 16, 0)}),
    ("diffusion9", (700, 700), 16, {"tile": (4, 0, 0)}),
    ("jacobi2d", (9000, 40), 40, {"tile": (0, 16, 0)}),
    ("cloudsim", (9000, 100), 20, {}),
])
def test_register_tiles(gpu, name, shape, n, kw):
    assert _run(name, shape, n, **kw) < -(-n // 4)
