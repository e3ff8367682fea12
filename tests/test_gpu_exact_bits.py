"""The exact solver's two face kernels give the same bits: two lanes a face where a context has at most 128 face chunks
(a simulation alone), one lane beyond (the same simulation beside a tube of 33,000 cells).  Which of them runs
depends on the whole context, so a batch's members may change from one to the other in the middle of a run."""
import dataclasses

import numpy as np
import pytest

from hydro_rs_amd import fvs, ics

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    if fvs.device_count() < 1:
        pytest.skip("no HIP device")


def _vortex(motion):
    p = ics.isentropic_vortex_2d(40, t_end=1.0)
    return dataclasses.replace(p, cfg=dataclasses.replace(p.cfg, solver=fvs.EXACT, motion=motion))


def _strong(n):
    """Shocks, rarefactions and near-vacuum of a random tube: every branch of the pressure iteration."""
    rng = np.random.default_rng(3)
    p = ics.sod_1d(n, t_end=1.0)
    k = n // 8
    scale = np.repeat(10.0 ** rng.uniform(-2, 2, 8), [k] * 7 + [n - 7 * k])
    return dataclasses.replace(p, u_int=p.u_int * scale)


CASES = {"sod_fixed": lambda: ics.sod_1d(1000, t_end=1.0), "sod_moving": lambda: ics.sod_1d(1000, t_end=1.0, motion=fvs.FLUID),
         "strong": lambda: _strong(500), "vortex_fixed": lambda: _vortex(fvs.FIXED), "vortex_moving": lambda: _vortex(fvs.STEER)}


@pytest.mark.parametrize("precision", [fvs.FP64, fvs.FP32_FLUX])
@pytest.mark.parametrize("case", list(CASES))
def test_two_lanes_equal_one(case, precision):
    print(f"[exact bits] {case} precision {precision}", flush=True)
    prob = ics.with_precision(CASES[case](), precision)
    filler = ics.with_precision(ics.sod_1d(33000, t_end=1.0), precision)
    assert prob.cfg.solver == filler.cfg.solver == fvs.EXACT
    steps = 12
    alone, other, both = ics.build_device_sim(prob), ics.build_device_sim(filler), fvs.Batch.for_problems([prob, filler])
    assert alone.run(steps) == other.run(steps) == steps
    both.run(steps)
    ia, ib = alone.engine_info(), both.engine_info(0)
    assert ia["step_count"] == ib["step_count"] == steps and ia["face_fluxes"] == ib["face_fluxes"]
    a, b = alone.get_state(), both.get_state(0)
    for k in a:
        assert np.array_equal(a[k], b[k], equal_nan=a[k].dtype.kind == "f"), k
    assert both.stats()["brent_calls"] == alone.stats()["brent_calls"] + other.stats()["brent_calls"]
    for s in (alone, other, both):
        s.close()
