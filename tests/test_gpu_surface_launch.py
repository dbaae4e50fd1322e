"""GPU: the free-surface rows inside the PML sweep's launch and in one of their own.

On 32x8 tiles the rows ride with the sweep; per-launch timing runs them apart.
Both are the same update, so turning the timing on must not change a bit.
"""
import numpy as np
import pytest

import cgfd
from problem import Problem
from test_gpu_stage_forms import _vertical_lines

pytestmark = pytest.mark.gpu

STORE = {"f32": cgfd.STORE_F32, "f64": cgfd.STORE_F64}


def _grid(kind):
    kw = dict(ni=75, nj=37, nk=29, pml=(4, 5, 4, 3, 4, 0))
    if kind == "lines":
        return _vertical_lines(**kw)
    return Problem(curvilinear=kind == "curvilinear", hetero=0.05, seed=13, nt_total=10, init_random=True, **kw)


@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("split", [cgfd.SPLIT_PLANES, cgfd.SPLIT_CORE], ids=["planes", "core"])
@pytest.mark.parametrize("kind", ["cartesian", "lines", "curvilinear"])
def test_timed_run_equals_untimed_run(kind, split, storage):
    P = _grid(kind)
    out = []
    for timed in (False, True):
        s = cgfd.Session(P.ni, P.nj, P.nk, storage=STORE[storage])
        P.upload(s, dtype=np.float64 if storage == "f64" else np.float32)
        s.set_split(split)
        s.set_tile(1, 5)
        s.set_timing(timed)
        s.run(0, P.nt_total, P.dt)
        out.append(s.fetch_level(0, cgfd.LEVEL_PRE))
        s.close()
    assert np.array_equal(out[0], out[1])
