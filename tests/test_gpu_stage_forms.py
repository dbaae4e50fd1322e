"""GPU: the forms a stage takes, against the CPU oracle.

Sources reach a stage either from the table that the step's head writes over
each shot's box, or through a launch after the stage when their points spread
too far; runs are cut at odd steps, so both clocks of the head start a run.
The sum level of the last stage (FP32/FP64) is covered by every case.
Tolerances as in the parity tests: FP32 relative L2 <= 1e-5, FP64 <= 1e-11.
"""
import numpy as np
import pytest

import cgfd
from problem import Problem, rel_l2

pytestmark = pytest.mark.gpu

TOL = {"f32": 1e-5, "f64": 1e-11}
STORE = {"f32": cgfd.STORE_F32, "f64": cgfd.STORE_F64}


def _two_sources(a, b):
    """Both problems' sources as one table."""
    s, t = a.src, b.src
    out = dict(s, nsrc=2)
    for k in ("it_begin", "it_end", "ext_num", "ext_indx", "ext_coef"):
        out[k] = np.concatenate([s[k], t[k]])
    out["M"] = np.concatenate([s["M"], t["M"]], axis=1)
    a.src = out
    return a


def _problem(where, **kw):
    def make(ijk):
        return Problem(ni=37, nj=34, nk=30, curvilinear=True, hetero=0.05, seed=5, nt_total=19, init_random=True,
                       pml=(4, 4, 4, 4, 4, 0), src_ijk=ijk, **kw)
    if where == "far":   # a box of both would hold 24 x 20 x 7 points or more
        return _two_sources(make((8.2, 8.4, 12.1)), make((26.0, 24.7, 12.6)))
    if where == "near":  # one box, overlapping spreads
        return _two_sources(make((15.2, 14.4, 12.1)), make((17.0, 16.7, 13.6)))
    return make({"surface": (18.3, 15.0, 27.0), "pml": (3.0, 15.2, 12.0)}[where])


@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("where", ["near", "far", "surface", "pml"])
@pytest.mark.parametrize("split", ["planes", "shell", "core", "plain"])
def test_sources_in_every_split(split, where, storage):
    P = _problem(where)
    f = np.float64 if storage == "f64" else np.float32
    s = cgfd.Session(P.ni, P.nj, P.nk, storage=STORE[storage], flags=cgfd.FLAG_PLAIN if split == "plain" else 0)
    P.upload(s, dtype=f)
    if split != "plain":
        s.set_split({"planes": cgfd.SPLIT_PLANES, "shell": cgfd.SPLIT_SHELL, "core": cgfd.SPLIT_CORE}[split])
        s.set_tile(1, 4)
    s.run(0, 5, P.dt)
    s.run(5, 1, P.dt)
    s.run(6, 13, P.dt)
    seis, wave = s.read_seismo(0), s.fetch_level(0, cgfd.LEVEL_PRE)
    s.close()
    so, wo, _ = P.oracle_run(64 if storage == "f64" else 32)
    assert rel_l2(seis, so) <= TOL[storage]
    for c in range(9):
        assert rel_l2(wave[c], wo[c]) <= TOL[storage], c


@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("shape", [0, 1], ids=["own-launch", "with-sweep"])
@pytest.mark.parametrize("ni,nj", [(32, 24), (33, 25), (31, 40), (65, 23)])
def test_surface_rows_at_tile_edges(ni, nj, shape, storage):
    P = Problem(ni=ni, nj=nj, nk=24, curvilinear=True, hetero=0.05, seed=9, nt_total=9, init_random=True,
                pml=(4, 4, 4, 4, 4, 0))
    f = np.float64 if storage == "f64" else np.float32
    s = cgfd.Session(P.ni, P.nj, P.nk, storage=STORE[storage])
    P.upload(s, dtype=f)
    s.set_tile(shape, 8)
    s.run(0, P.nt_total, P.dt)
    wave = s.fetch_level(0, cgfd.LEVEL_PRE)
    s.close()
    _, wo, _ = P.oracle_run(64 if storage == "f64" else 32)
    for c in range(9):
        assert rel_l2(wave[c], wo[c]) <= TOL[storage], c
        assert rel_l2(wave[c][-7:-3], wo[c][-7:-3]) <= TOL[storage], c
