"""The Stencil methods put their result into output.hostArray whatever its memory
looks like (bit for bit the oracle's), and refuse what they cannot write."""
import numpy as np
import pytest

import oracle
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu
H, W, N = 33, 47, 6


def _unaligned():
    return np.zeros(H * W * 4 + 1, np.uint8)[1:].view(np.float32).reshape(H, W)


OUTPUTS = {
    "plain": lambda: np.zeros((H, W), np.float32),
    "double": lambda: np.zeros((H, W), np.float64),
    "strided": lambda: np.zeros((H, 2 * W), np.float32)[:, ::2],
    "fortran": lambda: np.zeros((H, W), np.float32, order="F"),
    "unaligned": _unaligned,
    "subclass": lambda: np.ma.array(np.zeros((H, W), np.float32)),
}


def _stencil(out):
    a = inputs.uniform(3, 0, H * W).reshape(H, W)
    src, dst = api.Array2D(W, H), api.Array2D(W, H)
    src.hostArray[...] = a
    out[...] = a
    dst.hostArray = out
    return a, api.Stencil2D(src, dst, api.Mask2D(4), K.jacobi2d())


@pytest.mark.parametrize("kind", list(OUTPUTS))
def test_result_lands_in_the_output_array(gpu, kind):
    out = OUTPUTS[kind]()
    a, st = _stencil(out)
    st.runIterativeGPU(N)
    want = oracle.run_2d(K.jacobi2d(), a, N)
    assert st.output.hostArray is out
    assert np.array_equal(np.asarray(out, np.float32).view(np.uint32), want.view(np.uint32))


def test_outputs_that_are_refused(gpu):
    out = np.zeros((H, W), np.float32)
    a, st = _stencil(out)
    out.flags.writeable = False
    with pytest.raises(ValueError):
        st.runIterativeGPU(N)
    assert np.array_equal(out, a)
    _, st = _stencil(np.zeros((H, W), np.int32))
    with pytest.raises(TypeError):
        st.runIterativeGPU(N)
