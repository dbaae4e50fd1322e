"""GPU: the bare right-hand side under every pinned tile shape against the oracle
(FP32 relative L2 <= 1e-5 per component, FP64 <= 1e-11)."""
import numpy as np
import pytest

import cgfd
from problem import Problem, rel_l2

pytestmark = pytest.mark.gpu

STORE = {"f32": (cgfd.STORE_F32, np.float32, 32, 1e-5), "f64": (cgfd.STORE_F64, np.float64, 64, 1e-11)}


@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("shape,zchunk", [(0, 5), (1, 48), (2, 7), (3, 4)])
@pytest.mark.parametrize("curv", [False, True], ids=["cart", "curv"])
def test_onestage_on_each_tile(curv, shape, zchunk, storage):
    st, f, prec, tol = STORE[storage]
    P = Problem(ni=75, nj=37, nk=29, curvilinear=curv, pml=(4, 5, 4, 3, 4, 0), hetero=0.05, init_random=True, nt_total=6,
                seed=3)
    s = cgfd.Session(P.ni, P.nj, P.nk, storage=st)
    P.upload(s, dtype=f)
    s.set_tile(shape, zchunk)
    for pair, stage in ((0, 0), (2, 1), (5, 3)):
        s.onestage(0, cgfd.LEVEL_PRE, pair, stage, 3)
        got = s.fetch_level(0, cgfd.LEVEL_RHS)
        want, _ = P.oracle_stage(P.init, pair, stage, 3, precision=prec)
        for c in range(9):
            assert rel_l2(got[c], want[c]) <= tol, (pair, stage, c)
    s.close()
