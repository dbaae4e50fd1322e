"""GPU: the metric components a sweep or a surface row may leave out.

What is dropped must lie below the rounding of the session's own arithmetic:
against the form that streams every component (FLAG_FULL_METRIC) nothing may
change where the noise is larger than that, and the right-hand side is then
equal bit for bit.
"""
import numpy as np
import pytest

import cgfd
from problem import Problem
from test_gpu_stage_forms import _vertical_lines

pytestmark = pytest.mark.gpu

STORE = {"f32": cgfd.STORE_F32, "f64": cgfd.STORE_F64}


def _rhs(P, storage, flags=0):
    f = np.float64 if storage == "f64" else np.float32
    s = cgfd.Session(P.ni, P.nj, P.nk, storage=STORE[storage], flags=flags)
    P.upload(s, dtype=f)
    s.set_tile(1, 6)
    out = []
    for pair, stage in ((0, 0), (2, 1)):
        s.onestage(0, cgfd.LEVEL_PRE, pair, stage, 0)
        out.append(s.fetch_level(0, cgfd.LEVEL_RHS))
    const = s.const_metric()
    s.close()
    return np.stack(out), const


def _noise(P, comp, size):
    rng = np.random.default_rng(comp)
    P.metric[comp] += size * rng.choice([-1.0, 1.0], P.metric[comp].shape)
    return P


@pytest.mark.parametrize("storage,size", [("f64", 5e-13), ("f64", 2e-14), ("f32", 1e-6)])
@pytest.mark.parametrize("comp", [1, 2, 5, 6])
def test_vertical_lines_with_noise_above_rounding_keep_the_arrays(comp, storage, size):
    P = _noise(_vertical_lines(ni=40, nj=30, nk=24, pml=(3, 3, 3, 3, 3, 0)), comp, 0.01 * size)
    auto, const = _rhs(P, storage)
    full, _ = _rhs(P, storage, cgfd.FLAG_FULL_METRIC)
    assert not const
    assert np.array_equal(auto, full)


@pytest.mark.parametrize("comp", [2, 4])
def test_tolerance_follows_the_rows_own_scale(comp):
    """Cells far wider than high: the xi and eta rows are small beside zeta's."""
    P = _vertical_lines(ni=40, nj=30, nk=24, pml=(3, 3, 3, 3, 3, 0))
    P.metric[1] *= 1e-2
    P.metric[5] *= 1e-2
    P.metric[7:10] *= 1e2
    P = _noise(P, comp, 5e-11)   # 5e-7 of xi_x or eta_y, 5e-11 of zeta_z
    auto, const = _rhs(P, "f32")
    full, _ = _rhs(P, "f32", cgfd.FLAG_FULL_METRIC)
    assert not const
    assert np.array_equal(auto, full)


@pytest.mark.parametrize("comp", [1, 2, 7, 9])
def test_surface_rows_of_a_nearly_cartesian_fp64_grid_keep_the_arrays(comp):
    P = Problem(ni=40, nj=30, nk=24, hetero=0.05, seed=13, init_random=True, pml=(3, 3, 3, 3, 3, 0))
    P.metric[:] = 0.0
    P.metric[0], P.metric[1], P.metric[5], P.metric[9] = 1e6, 0.01, 0.01, 0.01
    P = _noise(P, comp, 0.01 * 3e-11)
    auto, const = _rhs(P, "f64")
    full, _ = _rhs(P, "f64", cgfd.FLAG_FULL_METRIC)
    assert const
    rows = slice(3 + P.nk - 4, 3 + P.nk)
    assert np.array_equal(auto[:, :, rows], full[:, :, rows])
