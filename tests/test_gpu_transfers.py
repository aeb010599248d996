"""Uploads and downloads of grids whose rows are shorter than their pitch: host
rows cross the link packed and a kernel spreads or gathers them, in the widest
unit (1 to 16 bytes) that divides a row.  A copy, so every value is equal."""
import numpy as np
import pytest

from pskel_amd import api

pytestmark = pytest.mark.gpu

# rows of odd bytes, of 2, 4, 8 and 16-byte multiples, whole pitches, single
# cells, more rows in a chunk than grid rows of a launch (90000 x 200), several
# 16 MiB chunks (the last one ragged)
CASES = [("u8", (7, 1)), ("u8", (1000, 1503)), ("u8", (33, 1024)), ("u8", (5, 17000)), ("u8", (90000, 200)),
         ("u8", (20011, 1999)), ("f32", (3, 1)), ("f32", (501, 257)), ("f32", (77, 130)), ("f32", (64, 256)),
         ("f32", (4099, 2051)), ("f32", (6, 5, 3)), ("f32", (150, 41, 211)), ("bf16", (5, 7, 3)), ("bf16", (9, 5, 1030)),
         ("f16", (40, 33, 66))]


@pytest.mark.parametrize("storage,shape", CASES)
def test_pitched_rows_round_trip(gpu, storage, shape):
    r = np.random.default_rng(sum(shape))
    if storage in ("bf16", "f16"):  # raw storage words
        mk = lambda: r.integers(0, 1 << 16, shape, dtype=np.uint16)  # noqa: E731
    elif storage == "u8":
        mk = lambda: r.integers(0, 2, shape, dtype=np.uint8)  # noqa: E731
    else:
        mk = lambda: r.standard_normal(shape, dtype=np.float32)  # noqa: E731
    a, b = mk(), mk()
    raw = storage in ("bf16", "f16")
    with api.Grid(shape, storage) as g:
        g.upload(0, a)
        g.upload(1, b)
        assert np.array_equal(g.download(raw=raw).view(np.uint8), a.view(np.uint8))
        assert np.array_equal(g.download_previous(raw=raw).view(np.uint8), b.view(np.uint8))
        g.upload(0, b)  # the staging buffers once more
        assert np.array_equal(g.download(raw=raw).view(np.uint8), b.view(np.uint8))
