"""Whose model answers for stencils that the shipped model was not trained on (field
stencils, masks without a specialised kernel): a model the caller passes or installs
does; the shipped one leaves them to the heuristic, however it was loaded."""
import ctypes as C
import os

import numpy as np
import pytest

from pskel_amd import _lib as L
from pskel_amd import kernels as K
from pskel_amd import tuner as T

pytestmark = pytest.mark.gpu

SKEW3 = [(0, 0), (1, 0), (0, 2)]


def _queries():
    q = L.TuneQuery()
    q.ndim, q.storage, q.height, q.width, q.depth, q.iterations = 2, T.STORAGE["f32"], 700, 1100, 1, 20
    for s in (K.cloudsim(0.01), K.Stencil(K.WEIGHTED_SUM, 2, SKEW3, weights=[0.5, 0.25, 0.25])):
        yield q, s.desc()


def _candidates(q, d):
    buf, n = (L.LaunchCfg * L.TUNER_MAX_CANDIDATES)(), C.c_size_t()
    L.check(L.lib().pskel_tuner_candidates(C.byref(q), C.byref(d), buf, L.TUNER_MAX_CANDIDATES, C.byref(n)))
    X = np.zeros((n.value, L.TUNER_NFEAT), np.float32)
    for i in range(n.value):
        L.check(L.lib().pskel_tuner_features(C.byref(q), C.byref(d), C.byref(buf[i]),
                                             X[i].ctypes.data_as(C.POINTER(C.c_float))))
    return [T.cfg_key(buf[i]) for i in range(n.value)], X


def _choose(handle, q, d):
    out = L.LaunchCfg()
    L.check(L.lib().pskel_tuner_choose(handle, C.byref(q), C.byref(d), C.byref(out)))
    return T.cfg_key(out)


def _heuristic(q, d):
    out = L.LaunchCfg()
    L.check(L.lib().pskel_tuner_heuristic(C.byref(q), C.byref(d), C.byref(out)))
    return T.cfg_key(out)


def _close(m):
    m.close()  # and its place as the default
    if T.default_model() is not None:
        T.default_model().install()


def test_callers_model_answers(gpu):
    differs = 0
    for seed in (1, 2, 3):
        m = T.CostModel(seed=seed)
        try:
            for q, d in _queries():
                keys, X = _candidates(q, d)
                want = keys[int(np.argmin(m.predict(X)))]
                assert _choose(m._h, q, d) == want
                differs += want != _heuristic(q, d)
                m.install()
                assert _choose(None, q, d) == want
        finally:
            _close(m)
    assert differs  # untrained models do not agree with the heuristic throughout


@pytest.mark.skipif(not os.path.exists(T.DEFAULT_MODEL), reason="no shipped cost model")
def test_shipped_model_leaves_them_to_the_heuristic(gpu):
    m = T.CostModel.load()
    try:
        for q, d in _queries():
            assert _choose(m._h, q, d) == _heuristic(q, d)
            m.install()
            assert _choose(None, q, d) == _heuristic(q, d)
    finally:
        _close(m)
