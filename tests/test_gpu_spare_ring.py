"""Runs of different mask ranges on one grid.  Even fused depths write a spare
buffer, which holds the ring of the current state: as many rows and columns as
the range of the sweeps that write it, however narrow the ring of the runs before.
Single sweeps between the runs leave both states of the ping-pong pair as the
oracle has them, so every run is bit-equal to the oracle's from there."""
import numpy as np
import pytest

import oracle
from pskel_amd import api, inputs
from pskel_amd import kernels as K

pytestmark = pytest.mark.gpu


def _wide(radius):
    s = K.jacobi2d()
    s.radius = radius  # a mask range above the farthest offset: a ring of `radius` cells
    return s


def _check(g, want, what):
    assert np.array_equal(g.download().view(np.uint32), want.view(np.uint32)), what


@pytest.mark.parametrize("radius", [2, 3])
@pytest.mark.parametrize("use_graph", [False, True])
def test_wider_range_after_fused_runs(gpu, radius, use_graph):
    a = inputs.uniform(71, 0, 90 * 300).reshape(90, 300)
    b = a.copy()
    b[0, :], b[-1, :], b[:, 0], b[:, -1] = 3.0, -2.0, 0.5, 7.0
    narrow, wide = K.jacobi2d(), _wide(radius)
    cur, prev = a, b
    with api.Grid(a.shape, "f32") as g:
        g.upload_pair(a, b)
        for rep in range(3):
            # fused at range 1, then two single sweeps: the spare's parity is the
            # current state's, its inner rows are those of an older state
            g.run(narrow, 8, variant="tuned", time_tile=4, use_graph=use_graph)
            g.run(narrow, 2, variant="tuned", use_graph=use_graph)
            cur, prev = oracle.run_2d(narrow, cur, 10, out=prev), oracle.run_2d(narrow, cur, 9, out=prev)
            _check(g, cur, ("narrow", rep))
            # fused at the wide range, then two single sweeps again
            g.run(wide, 4, variant="tuned", time_tile=4, use_graph=use_graph)
            g.run(wide, 2, variant="tuned", use_graph=use_graph)
            api.synchronize()
            cur, prev = oracle.run_2d(wide, cur, 6, out=prev), oracle.run_2d(wide, cur, 5, out=prev)
            _check(g, cur, ("wide", rep))


def test_wider_range_after_a_batch(gpu):
    """The batch's sweeps write the same buffers at their own range."""
    a = inputs.uniform(72, 0, 64 * 200).reshape(64, 200)
    narrow, wide = K.jacobi2d(), _wide(2)
    with api.Grid(a.shape, "f32") as g:
        g.upload_pair(a)
        g.run(wide, 4, variant="tuned", time_tile=4)
        g.run(wide, 2, variant="tuned")
        with api.Batch([g], [narrow]) as batch:
            batch.run(2)
        cur, prev = oracle.run_2d(wide, a, 6), oracle.run_2d(wide, a, 5)
        cur, prev = oracle.run_2d(narrow, cur, 2, out=prev), oracle.run_2d(narrow, cur, 1, out=prev)
        _check(g, cur, "batch")
        g.run(wide, 4, variant="tuned", time_tile=4)
        _check(g, oracle.run_2d(wide, cur, 4, out=prev), "after the batch")


def test_ring_written_between_runs(gpu):
    """pskel_grid_swap: the caller's own sweep wrote the other buffer, its ring
    included (here: an upload of another state with another ring)."""
    from pskel_amd import _lib as L

    a = inputs.uniform(73, 0, 64 * 200).reshape(64, 200)
    s = K.jacobi2d()
    with api.Grid(a.shape, "f32") as g:
        g.upload_pair(a)
        g.run(s, 8, variant="tuned", time_tile=4)  # the spare exists
        info = g.info()
        for value in (5.0, -5.0):
            # the caller's sweep: a whole buffer of `value` into the previous state
            host = np.full((64, info["pitch"]), value, np.float32)
            L.check(L.lib().pskel_memcpy(g.info()["previous"], host.ctypes.data, host.nbytes, 1))
            L.check(L.lib().pskel_grid_swap(g._h))
        cur = np.full(a.shape, -5.0, np.float32)
        g.run(s, 8, variant="tuned", time_tile=4)
        _check(g, oracle.run_2d(s, cur, 8, out=np.full(a.shape, 5.0, np.float32)), "swap")
