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
STORE16 = {"f16": cgfd.STORE_F16, "bf16": cgfd.STORE_BF16}


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


def _vertical_lines(**kw):
    """A problem on evenly spaced vertical lines: xi_x and eta_y constant, the
    other xi and eta terms zero, zeta varying in every direction."""
    P = Problem(curvilinear=False, hetero=0.05, seed=13, nt_total=10, init_random=True, **kw)
    kk, jj, ii = np.meshgrid(*(np.arange(n) - 3.0 for n in (P.nz, P.ny, P.nx)), indexing="ij")
    s = (kk + 3.0) / P.nz
    z_i, z_j = 9.0 * s * np.cos(0.21 * ii + 0.1 * jj), -7.0 * s * np.sin(0.17 * jj + 0.05 * ii)
    z_k = 100.0 + 12.0 * np.sin(0.09 * ii) * np.cos(0.11 * jj) + 8.0 * s
    m = np.zeros_like(P.metric)
    m[0] = 1e4 * z_k
    m[1], m[5] = 0.01, 0.01
    m[7], m[8], m[9] = -0.01 * z_i / z_k, -0.01 * z_j / z_k, 1.0 / z_k
    P.metric = np.float64(np.float32(m))
    if P.free_top:
        P.mvx, P.mvy = (np.float64(np.float32(v)) for v in cgfd.free_surface_matrices(
            P.ni, P.nj, P.nk, P.metric, P.lam, P.mu))
    return P


def _run(P, storage, flags=0, split=None, tile=None):
    f = np.float64 if storage == "f64" else np.float32
    s = cgfd.Session(P.ni, P.nj, P.nk, storage=STORE[storage], flags=flags)
    P.upload(s, dtype=f)
    if split is not None:
        s.set_split(split)
    s.set_tile(*tile)
    s.run(0, P.nt_total, P.dt)
    out = s.fetch_level(0, cgfd.LEVEL_PRE)
    assert not s.const_metric()
    s.close()
    return out


@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("tile", [(0, 5), (1, 2), (1, 3), (2, 7)], ids=["64x4", "32x8/2", "32x8/3", "64x8"])
@pytest.mark.parametrize("split", [cgfd.SPLIT_PLANES, cgfd.SPLIT_CORE, cgfd.SPLIT_SHELL],
                         ids=["planes", "core", "shell"])
@pytest.mark.parametrize("free", [True, False], ids=["free", "pml"])
def test_vertical_line_metric(free, split, tile, storage):
    P = _vertical_lines(ni=75, nj=37, nk=29, free_top=free, pml=(4, 5, 4, 3, 4, 0 if free else 5))
    got = _run(P, storage, split=split, tile=tile)
    full = _run(P, storage, flags=cgfd.FLAG_FULL_METRIC, split=split, tile=tile)
    _, wo, _ = P.oracle_run(64 if storage == "f64" else 32)
    for c in range(9):
        assert rel_l2(got[c], wo[c]) <= TOL[storage], c
        # the same sums in another order: 40 stages at one or two roundings each
        assert rel_l2(got[c], full[c]) <= (1e-13 if storage == "f64" else 1e-5), c


@pytest.mark.parametrize("storage,off", [("f32", 1e-6), ("f64", 1e-11)])
@pytest.mark.parametrize("comp", [1, 2, 6])
def test_uneven_lines_keep_the_metric_arrays(comp, storage, off):
    """One xi or eta value beyond the tolerance: every component is streamed."""
    P = _vertical_lines(ni=40, nj=30, nk=24, pml=(3, 3, 3, 3, 3, 0))
    P.metric[comp, 11, 12, 13] += 0.01 * off
    a = _run(P, storage, tile=(1, 6))
    b = _run(P, storage, flags=cgfd.FLAG_FULL_METRIC, tile=(1, 6))
    assert np.array_equal(a, b)


@pytest.mark.parametrize("storage", ["f16", "bf16"])
@pytest.mark.parametrize("nk", [12, 29])
def test_16bit_tuned_form_is_bit_identical(nk, storage):
    """What tuning picks equals the plainest pinned form of the same split class."""
    P = Problem(ni=75, nj=37, nk=nk, hetero=0.05, seed=13, nt_total=6, init_random=True, pml=(4, 5, 4, 3, 4, 0))
    out, cls = [], None
    for pinned in (False, True):
        s = cgfd.Session(P.ni, P.nj, P.nk, storage=STORE16[storage])
        s.set_storage_scale(cgfd.storage_scales(STORE16[storage], P.ni, P.nj, P.nk, P.metric, P.lam, P.mu, P.slw,
                                                P.src, P.dt))
        P.upload(s)
        if pinned:
            s.set_split(cgfd.SPLIT_SHELL if cls == cgfd.SPLIT_SHELL else cgfd.SPLIT_PLANES)
            s.set_tile(1, 8)
        s.run(0, P.nt_total, P.dt)
        cls = s.get_split()
        out.append(s.fetch_level(0, cgfd.LEVEL_PRE))
        s.close()
    assert np.isfinite(out[0]).all()
    assert np.array_equal(out[0], out[1])
