"""CLOUDSIM on a device with no room for the spare buffer of fused sweeps: it runs in
single sweeps, as it does when no depth is named."""
import ctypes as C

import numpy as np
import pytest

from pskel_amd import _lib as L
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _alloc(nbytes):
    p = C.c_void_p()
    return p if L.lib().pskel_device_alloc(nbytes, C.byref(p)) == 0 else None


def test_cloudsim_without_room_for_a_spare(gpu):
    h = w = 8192  # a buffer is 256 MiB
    t = (np.float32(15.0) + np.float32(10.0) * inputs.uniform(3, 0, h * w)).reshape(h, w)
    wx = (inputs.uniform(4, 0, h * w) - np.float32(0.5)).reshape(w, h)
    s = K.cloudsim(0.01)
    held = []
    with api.Grid((h, w), "f32") as g, api.Field(wx) as fx, api.Field(-wx) as fy:
        for i, f in enumerate((fx, fy)):
            g.set_field(i, f)
        g.upload_pair(t)
        g.run(s, 7, variant="tuned", residual_every=7)
        want, previous = g.download(), g.download_previous()
        g.upload_pair(t)
        try:
            reserve = _alloc(64 * MIB)
            assert reserve
            for step in (16384 * MIB, 1024 * MIB, 128 * MIB):
                while len(held) < 1000:
                    p = _alloc(step)
                    if not p:
                        break
                    held.append(p)
            L.lib().pskel_device_free(reserve)
            # between 64 and 192 MiB are free: no third buffer
            st = g.run(s, 7, variant="tuned", time_tile=4, residual_every=7)
            assert st["launches"] == 7
            got, before = g.download(), g.download_previous()
        finally:
            for p in held:
                L.lib().pskel_device_free(p)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        assert np.array_equal(before.view(np.uint32), previous.view(np.uint32))
        # with the memory back, the next run fuses
        g.upload_pair(t)
        assert g.run(s, 7, variant="tuned", time_tile=4)["launches"] < 7
        assert np.array_equal(g.download().view(np.uint32), want.view(np.uint32))
