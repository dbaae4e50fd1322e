"""GPU: a shot's result does not depend on the sources of its batch companions.

Shots with a compact source (its rates join the stages), with sources that
spread too far for a table (a launch after each stage) and with none share one
session; each must equal its own single-shot run bit for bit, also when the
wide one is admitted while the others run.
"""
import numpy as np
import pytest

import cgfd
from problem import Problem, rel_l2

pytestmark = pytest.mark.gpu

STORE = {"f32": cgfd.STORE_F32, "f64": cgfd.STORE_F64, "f16": cgfd.STORE_F16}
TOL = {"f32": 1e-5, "f64": 1e-11}
DT = {"f32": np.float32, "f64": np.float64, "f16": np.float32}


def _shot(nt, *places):
    """One model for every call (same seed); the sources at `places` as one table."""
    ps = [Problem(ni=37, nj=34, nk=30, curvilinear=True, hetero=0.05, seed=5, nt_total=nt, init_random=True,
                  pml=(4, 4, 4, 4, 4, 0), src_ijk=q) for q in (places or [None])]
    P = ps[0]
    if not places:
        P.src = None
    elif len(ps) > 1:
        src = [p.src for p in ps]
        P.src = dict(src[0], nsrc=len(src), M=np.concatenate([s["M"] for s in src], axis=1))
        for k in ("it_begin", "it_end", "ext_num", "ext_indx", "ext_coef"):
            P.src[k] = np.concatenate([s[k] for s in src])
    return P


def _compact(nt):
    return _shot(nt, (15.2, 14.4, 12.1))


def _wide(nt):   # a box of both would hold 24 x 23 x 7 points
    return _shot(nt, (8.2, 8.4, 12.1), (26.0, 24.7, 12.6))


def _near(nt):   # a larger box than _compact's
    return _shot(nt, (15.2, 14.4, 12.1), (17.0, 16.7, 13.6))


def _session(P, storage, nshots, split):
    s = cgfd.Session(P.ni, P.nj, P.nk, storage=STORE[storage], nshots=nshots)
    if storage == "f16":
        s.set_storage_scale([-3] * 3 + [20] * 6)
    P.upload(s, shots=[], dtype=DT[storage])
    s.set_split(split)
    s.set_tile(1, 6)
    return s


def _alone(P, storage, split):
    s = _session(P, storage, 1, split)
    P.upload_shot(s, 0, DT[storage])
    s.run(0, P.nt_total, P.dt)
    out = s.read_seismo(0), s.fetch_level(0, cgfd.LEVEL_PRE)
    s.close()
    return out


def _check(s, shot, ref):
    assert np.array_equal(s.read_seismo(shot), ref[0]), shot
    assert np.array_equal(s.fetch_level(shot, cgfd.LEVEL_PRE), ref[1]), shot


@pytest.mark.parametrize("storage", ["f32", "f64", "f16"])
@pytest.mark.parametrize("split", [cgfd.SPLIT_PLANES, cgfd.SPLIT_SHELL], ids=["planes", "shell"])
def test_each_shot_of_a_mixed_batch_equals_its_own_run(split, storage):
    shots = [_compact(19), _wide(19), _near(19), _shot(19)]
    refs = [_alone(P, storage, split) for P in shots]
    if storage in TOL:
        for P, r in zip(shots[:3], refs):
            assert rel_l2(r[0], P.oracle_run(64 if storage == "f64" else 32)[0]) <= TOL[storage]
    m = _session(shots[0], storage, len(shots), split)
    for n, P in enumerate(shots):
        P.upload_shot(m, n, DT[storage])
    m.run(0, 3, shots[0].dt)
    m.run(3, 16, shots[0].dt)
    for n, r in enumerate(refs):
        _check(m, n, r)
    m.close()


@pytest.mark.parametrize("storage", ["f32", "f64"])
def test_wide_source_admitted_mid_run(storage):
    A, B = _compact(32), _wide(16)
    split = cgfd.SPLIT_PLANES
    ra, rb = _alone(A, storage, split), _alone(B, storage, split)
    m = _session(A, storage, 2, split)
    A.upload_shot(m, 0, DT[storage])
    m.set_shot(1, False)
    m.run(0, 16, A.dt)
    m.reset_shot(1)
    B.upload_shot(m, 1, DT[storage])
    m.set_shot(1, True, 16)
    m.run(16, 16, A.dt)
    _check(m, 0, ra)
    _check(m, 1, rb)
    m.close()
