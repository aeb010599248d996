"""The shipped model's timings hold no tall grids of one tile's width: the 9-point stencil
takes its rows there from measured lines, at both sides of each."""
import pytest

from pskel_amd import kernels as K
from pskel_amd import tuner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,rows", [((3501, 120), 8), ((14000, 1), 8), ((14001, 20), 16), ((24000, 60), 16),
                                        ((24001, 60), 32), ((32000, 9), 32), ((32001, 120), 16), ((1000000, 2), 16)])
@pytest.mark.parametrize("iterations", [2, 3, 60])
def test_rows(gpu, shape, rows, iterations):
    cfg = tuner.choose_config(K.diffusion9(), shape, "f32", iterations)
    assert cfg["variant"] == "tuned" and cfg["time_tile"] == min(iterations, 4) and tuple(cfg["tile"]) == (0, rows, 0)

