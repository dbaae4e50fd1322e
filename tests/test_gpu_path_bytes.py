"""GPU: the bench line's own-bytes figure follows the metric words the sweep loads."""
import os
import sys

import numpy as np
import pytest

import cgfd
from problem import Problem
from test_gpu_stage_forms import _vertical_lines

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402

pytestmark = pytest.mark.gpu

STORE = {"f32": cgfd.STORE_F32, "f64": cgfd.STORE_F64, "f16": cgfd.STORE_F16}


def _grid(kind):
    kw = dict(ni=40, nj=30, nk=24, pml=(3, 3, 3, 3, 3, 0))
    if kind == "lines":
        return _vertical_lines(**kw)
    P = Problem(curvilinear=kind == "sheared", nt_total=4, **kw)
    if kind == "cartesian":
        P.metric[:] = 0.0
        P.metric[0], P.metric[1], P.metric[5], P.metric[9] = 1e6, 0.01, 0.01, 0.01
    return P


@pytest.mark.parametrize("storage,shape,kind,words,nbytes", [
    ("f32", 1, "cartesian", 0, 120), ("f32", 0, "lines", 3, 132), ("f32", 1, "lines", 3, 132),
    ("f32", 2, "lines", 9, 156), ("f32", 1, "sheared", 9, 156), ("f64", 1, "lines", 3, 264),
    ("f64", 3, "lines", 9, 312), ("f16", 1, "lines", 9, 106.5), ("f16", 1, "cartesian", 0, 70.5)])
def test_metric_words_and_path_bytes(storage, shape, kind, words, nbytes):
    P = _grid(kind)
    s = cgfd.Session(P.ni, P.nj, P.nk, storage=STORE[storage])
    P.upload(s, shots=[], dtype=np.float64 if storage == "f64" else np.float32)
    s.set_tile(shape, 8)
    got = s.metric_words()
    s.close()
    assert got == words
    assert bench.path_bytes(storage, got) == nbytes
