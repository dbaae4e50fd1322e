"""GPU: a wavefield with no rates keeps its bits.

In a medium of zero stiffness and zero buoyancy every right-hand side is zero,
so W^{n+1} = W^n exactly: every level a step stores then holds W, whatever the
RK weights round to.  A combination that scales W before it is stored rounds
it, and the error grows with every step.
"""
import numpy as np
import pytest

import cgfd
from problem import Problem

pytestmark = pytest.mark.gpu

STORE = {"f32": cgfd.STORE_F32, "f64": cgfd.STORE_F64, "f16": cgfd.STORE_F16, "bf16": cgfd.STORE_BF16}


@pytest.mark.parametrize("storage", sorted(STORE))
@pytest.mark.parametrize("split", ["planes", "shell", "core", "plain"])
def test_zero_rates_keep_the_field(split, storage):
    P = Problem(ni=75, nj=37, nk=29, curvilinear=True, seed=4, init_random=True, nt_total=11, source=None,
                pml=(4, 5, 4, 3, 4, 0))
    for a in (P.lam, P.mu, P.slw):
        a[...] = 0.0
    s = cgfd.Session(P.ni, P.nj, P.nk, storage=STORE[storage], flags=cgfd.FLAG_PLAIN if split == "plain" else 0)
    if storage == "f16":
        s.set_storage_scale([-3] * 3 + [20] * 6)
    P.upload(s, dtype=np.float64 if storage == "f64" else np.float32)
    if split != "plain":
        s.set_split({"planes": cgfd.SPLIT_PLANES, "shell": cgfd.SPLIT_SHELL, "core": cgfd.SPLIT_CORE}[split])
        s.set_tile(1, 6)
    before = s.fetch_level(0, cgfd.LEVEL_PRE)
    s.run(0, P.nt_total, P.dt)
    after = s.fetch_level(0, cgfd.LEVEL_PRE)
    s.close()
    assert np.abs(before).max() > 0
    assert np.array_equal(after, before)
