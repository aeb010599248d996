"""Which kernel a run of an arbitrary mask takes: the LDS tile on full volumes, the
plain kernel where most tile cells lie outside a thin grid or most cells are copied
faces (there the tile measured 2 to 16 times slower)."""
import ctypes as C
import itertools

import pytest

import shapes
from pskel_amd import kernels as K

BOX27 = list(itertools.product((-1, 0, 1), repeat=3))
STAR7 = [(0, 0, 0)] + [tuple(s if i == j else 0 for j in range(3)) for i in range(3) for s in (-1, 1)]
ROW17 = [(0, 0, i) for i in range(-8, 9)]


def _pays(offs, shape, boundary=K.BOUNDARY_COPY, half=0, block=(64, 4)):
    l = shapes.lib()
    s = K.Stencil(K.WEIGHTED_SUM, len(shape), offs, weights=[1.0 / len(offs)] * len(offs), boundary=boundary)
    d = s.desc()
    h, w, dd = shape if len(shape) == 3 else (*shape, 1)
    return bool(l.shapes_points_pay(C.byref(d), len(shape), w, h, dd, half, *block))


@pytest.mark.parametrize("half", [0, 1])
@pytest.mark.parametrize("boundary", [K.BOUNDARY_COPY, K.BOUNDARY_HALO])
def test_volumes_take_the_tile(boundary, half):
    for shape in ((128, 128, 128), (192, 225, 260), (256, 256, 256)):
        for offs in (BOX27, STAR7):
            assert _pays(offs, shape, boundary, half), (shape, len(offs))
    assert _pays([(i, j) for i in range(-2, 3) for j in range(-2, 3)], (2048, 2048))


@pytest.mark.parametrize("half", [0, 1])
def test_thin_grids_take_the_plain_kernel(half):
    for offs in (BOX27, STAR7, ROW17):
        for shape in ((1, 1500, 1000), (2, 1000, 1000), (1000, 2, 1000), (1000, 1, 1000)):
            assert not _pays(offs, shape, K.BOUNDARY_COPY, half), (shape, len(offs))
    for offs in ([(0, 0), (0, 1)], [(i, j) for i in range(-3, 4) for j in range(-3, 4)]):
        assert not _pays(offs, (5, 200000)), len(offs)
    # no cell takes a sum
    assert not _pays(BOX27, (2, 600, 600), K.BOUNDARY_COPY, half)


def test_a_halo_that_does_not_fit():
    assert not _pays([(0, 0, -9), (0, 0, 0), (0, 0, 9)], (256, 256, 256), K.BOUNDARY_HALO)
