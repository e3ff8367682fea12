"""Fluxes computed by a trait-level call, to look at them, leave the engine's next steps what they were: a run after
hfv_compute_fluxes equals the run without it, bit for bit, and a simulation at its end takes no further step."""
import dataclasses

import numpy as np
import pytest

from hydro_rs_amd import _lib, fvs, ics

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    if fvs.device_count() < 1:
        pytest.skip("no HIP device")


def _next_info(sim):
    """TimestepInfo of the engine's next step."""
    e = sim.engine_info()
    return _lib.TimestepInfo(ti_old=e["ti_old"], ti_current=e["ti_next"], ti_next=e["ti_next"],
                             time_base=e["time_base"], time_base_inv=e["time_base_inv"])


def _pair(prob, steps):
    sims = [ics.build_device_sim(prob) for _ in range(2)]
    for s in sims:
        assert s.run(steps) == steps
    return sims


# dt_snap: with pending dump points (a step passes at most 8 of them) and without
@pytest.mark.parametrize("precision", [fvs.FP64, fvs.FP32_FLUX])
@pytest.mark.parametrize("make, dt_snap", [(lambda: ics.sedov_2d(side=24, t_end=0.01, seed=3), 0.0),
                                           (lambda: ics.sedov_2d(side=24, t_end=0.01, seed=3), 1e-4),
                                           (lambda: ics.kelvin_helmholtz_3d(side=8, t_end=0.2), 0.0),
                                           (lambda: ics.kelvin_helmholtz_3d(side=8, t_end=0.2), 1e-2)])
def test_run_after_compute_fluxes(make, dt_snap, precision):
    prob = ics.with_precision(make(), precision)
    prob = dataclasses.replace(prob, cfg=dataclasses.replace(prob.cfg, dt_snap=dt_snap))
    print(f"[phase then run] {prob.name} precision {precision} dt_snap {dt_snap}", flush=True)
    a, b = _pair(prob, 7)
    for steps in (1, 1, 9):
        a.compute_fluxes(_next_info(a))
        assert a.run(steps) == b.run(steps) == steps
        ia, ib = a.engine_info(), b.engine_info()
        assert ia == ib
        sa, sb = a.get_state(), b.get_state()
        for k in sb:
            assert np.array_equal(sa[k], sb[k]), (k, steps)


@pytest.mark.parametrize("precision", [fvs.FP64, fvs.FP32_FLUX])
def test_no_step_at_the_end(precision):
    print(f"[phase then run] end, precision {precision}", flush=True)
    sim = ics.build_device_sim(ics.with_precision(ics.sod_1d(100, t_end=0.01), precision))
    assert sim.run() > 0
    before, t = sim.get_state(), sim.engine_info()
    sim.compute_fluxes(_next_info(sim))
    assert sim.run(5) == 0
    assert sim.engine_info()["t_current"] == t["t_current"]
    after = sim.get_state()
    for k in before:
        assert np.array_equal(before[k], after[k]), k
