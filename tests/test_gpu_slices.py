"""Sliced gradient geometry (one slice per 64 cells, as long as its longest CSR row): bit for bit the per-step
geometry at ragged cell counts, with walls and periodic, staged neighbours or not, and the per-step path where a
slot's slices would not fit."""
import numpy as np
import pytest

from hydro_rs_amd import fvs, ics

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    if fvs.device_count() < 1:
        pytest.skip("no HIP device")


def _cloud(n, boundary, precision):
    """n uniformly random generators (cells of very unequal face counts), a pressure step along x."""
    loc = np.random.default_rng(n).uniform(0.0, 1.0, (n, 3))
    cfg = fvs.Config(dim=3, box=(1.0, 1.0, 1.0), gamma=5.0 / 3.0, cfl=0.3, solver=fvs.HLLC, boundary=boundary,
                     motion=fvs.FIXED, t_end=0.1, precision=precision)
    left = loc[:, 0] < 0.5
    return ics._finish("cloud3d", cfg, loc, np.where(left, 1.0, 0.5), np.zeros((n, 3)), np.where(left, 1.0, 0.3))


def _lattice(dim, side, precision):
    make = {1: lambda: ics.riemann_tube_1d(side, 1.0, 1.0, 0.0, 0.125, 0.1, 0.0, 1.4, t_end=0.1, precision=precision),
            2: lambda: ics.isentropic_vortex_2d(side, t_end=1.0, precision=precision),
            3: lambda: ics.kelvin_helmholtz_3d(side, t_end=1.0, precision=precision)}
    return make[dim]()


CASES = {"tube1d_3": lambda p: _lattice(1, 3, p), "tube1d_65": lambda p: _lattice(1, 65, p),
         "vortex2d_9": lambda p: _lattice(2, 9, p), "vortex2d_17": lambda p: _lattice(2, 17, p),
         "kh3d_3": lambda p: _lattice(3, 3, p), "kh3d_7": lambda p: _lattice(3, 7, p),
         "cloud3d_64_walls": lambda p: _cloud(64, fvs.REFLECTIVE, p),
         "cloud3d_300_open": lambda p: _cloud(300, fvs.OPEN, p)}


def _run(prob, static_grad, gstaged, steps=20):
    sim = ics.build_device_sim(prob)
    sim.set_tuning(0, -1, static_grad, gstaged)
    assert sim.tuning()["static_grad"] == static_grad
    sim.run(steps)
    out = sim.get_state()
    sim.close()
    return out


@pytest.mark.parametrize("precision", [fvs.FP64, fvs.FP32_FLUX])
@pytest.mark.parametrize("case", list(CASES))
def test_slices_equal_per_step_geometry(case, precision):
    print(f"[slices] {case} precision {precision}", flush=True)
    prob = CASES[case](precision)
    ref = _run(prob, 0, 0)
    for gstaged in (0, 1):
        got = _run(prob, 1, gstaged)
        for k in ref:
            assert np.array_equal(got[k], ref[k]), (k, gstaged)


def test_slices_that_do_not_fit_fall_back():
    """A batch slot of exact capacity holds 1.5 times its CSR entries in slices: a random cloud's need more, so
    it keeps the per-step geometry, with the results of a roomier slot that has the slices."""
    print("[slices] fallback", flush=True)
    prob = _cloud(1000, fvs.REFLECTIVE, fvs.FP64)
    tight, roomy = fvs.Batch.for_problems([prob]), fvs.Batch.for_problems([prob], headroom=2.0)
    assert tight.tuning(0)["static_grad"] == 0 and roomy.tuning(0)["static_grad"] == 1
    for b in (tight, roomy):
        b.run(12)
    a, b = tight.get_state(0), roomy.get_state(0)
    for k in a:
        assert np.array_equal(a[k], b[k]), k
