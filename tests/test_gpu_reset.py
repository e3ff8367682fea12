"""A slot that held another simulation is reset by one kernel before the next is loaded: runs in a reused slot equal
the same runs in a fresh batch, bit for bit, whatever either one's size and precision."""
import numpy as np
import pytest

from hydro_rs_amd import fvs, ics

pytestmark = pytest.mark.gpu

FIELDS = ["prim", "grad", "gc", "extrap", "cons", "fluxes", "v", "v_rel", "dt", "timebin"]


def _tube(n, seed, precision):
    return ics.riemann_tube_1d(n, 1.0, 1.0, 0.0, 0.125, 0.1, 0.0, 1.4, seed=seed, t_end=1.0, precision=precision)


@pytest.mark.parametrize("precision", [fvs.FP64, fvs.FP32_FLUX])
@pytest.mark.parametrize("n", [16, 255, 256, 257, 700])
def test_reused_slot_equals_fresh(n, precision):
    print(f"[reset] n={n} precision={precision}", flush=True)
    caps = [np.array([k], dtype=np.int64) for k in (800, 1000, 2000)]
    used, fresh = fvs.Batch(*caps), fvs.Batch(*caps)
    used.load(0, _tube(600, 1, precision))
    used.run(20)
    used.unload(0)
    for b in (used, fresh):
        b.load(0, _tube(n, 2, precision))
    for steps in (0, 12):
        for b in (used, fresh):
            if steps:
                b.run(steps)
        a, b = used.get_state(0, FIELDS), fresh.get_state(0, FIELDS)
        for k in FIELDS:
            assert np.array_equal(a[k], b[k]), (k, steps)
