"""GPU: what the autotuner may cost a session's first run, counted in its own steps.

Timing every choice three times over, small z chunks included, had made it about
990 steps in FP32 and 480 in FP16 on this model; it takes 380 and 220.
"""
import time

import pytest

import cgfd
import workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage,most", [(cgfd.STORE_F32, 640), (cgfd.STORE_F16, 320)], ids=["f32", "f16"])
def test_first_run_is_worth_few_steps(storage, most):
    w = workloads.small(ni=40, nj=36, nk=36, nt=8)     # the process's own start-up, outside the clock
    s = cgfd.Session(w["ni"], w["nj"], w["nk"], storage=storage)
    workloads.upload(s, w, nt_total=8)
    s.run(0, 1, w["dt"])
    s.close()
    m = workloads.small(ni=104, nj=96, nk=60, nt=80)   # a grid no other test has tuned
    s = cgfd.Session(m["ni"], m["nj"], m["nk"], storage=storage)
    workloads.upload(s, m, nt_total=80)
    t0 = time.perf_counter()
    s.run(0, 1, m["dt"])
    first = time.perf_counter() - t0
    s.run(1, 15, m["dt"])
    step = 1e30
    for it in range(16, 80, 16):
        t0 = time.perf_counter()
        s.run(it, 16, m["dt"])
        step = min(step, (time.perf_counter() - t0) / 16)
    s.close()
    print(f"first run {first * 1e3:.1f} ms, {first / step:.0f} steps of {step * 1e3:.3f} ms")
    assert first <= most * step
