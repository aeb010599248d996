"""The MLP's forward pass at input widths around the 16- and 4-wide parts of its
dot products, against the CPU oracle (FP64).  A sum of n f32 products of
standard-normal pairs is off by at most about n * 6e-8 of its terms' magnitudes:
1e-5 relative to 1 covers 33 of them and tanh."""
import ctypes as C

import numpy as np
import pytest

import oracle
from pskel_amd import _lib as L

pytestmark = pytest.mark.gpu
F = C.POINTER(C.c_float)


@pytest.mark.parametrize("nin", [1, 3, 4, 5, 15, 16, 17, 20, 33])
def test_mlp_forward_widths(gpu, nin):
    sizes = [nin, nin, 1]
    h, n = C.c_void_p(), C.c_size_t()
    L.check(L.lib().pskel_mlp_create((C.c_int32 * 3)(*sizes), 2, 7, 0, C.byref(h)))
    try:
        L.check(L.lib().pskel_mlp_num_params(h, C.byref(n)))
        p = np.zeros(n.value, np.float32)
        L.check(L.lib().pskel_mlp_get_params(h, p.ctypes.data_as(F), n.value))
        x = np.random.default_rng(nin).standard_normal((19, nin)).astype(np.float32)
        got = np.zeros(19, np.float32)
        L.check(L.lib().pskel_mlp_predict(h, x.ctypes.data_as(F), 19, got.ctypes.data_as(F)))
        np.testing.assert_allclose(got, oracle.mlp_predict(sizes, p, x.astype(np.float64)), rtol=1e-5, atol=1e-5)
    finally:
        L.lib().pskel_mlp_destroy(h)
