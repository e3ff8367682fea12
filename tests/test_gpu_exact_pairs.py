"""The exact solver's face kernel with two lanes a face (up to 128 face chunks) and with one (beyond): both against
the oracle after some steps, at the chunk and wave edges of either side, bins exact."""
import numpy as np
import pytest

from hydro_rs_amd import fvs, ics
from tests.helpers import oracle_sim, rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    if fvs.device_count() < 1:
        pytest.skip("no HIP device")


# cells of a tube with walls: cells + 1 faces; 31/32/33 a wave's pairs, 255/256 a chunk, 32767/33000 the rule
@pytest.mark.parametrize("n", [3, 30, 31, 32, 254, 255, 256, 1001, 32767, 33000])
@pytest.mark.parametrize("motion", [fvs.FIXED, fvs.FLUID])
def test_exact_pairs_match_oracle(ora, n, motion):
    print(f"[exact pairs] n={n} motion={motion}", flush=True)
    prob = ics.sod_1d(n, t_end=0.1, motion=motion)
    dev, ref = ics.build_device_sim(prob), oracle_sim(prob)
    steps = dev.run(6)
    assert ref.advance(steps) == steps
    got, want = dev.get_state(), ref.get_fields()
    assert np.array_equal(got["timebin"], want["timebin"])
    # the tolerance of whole runs: pow in the device libm may differ in its last bit, and steps compound it
    for k in ("prim", "cons"):
        assert rel_err(got[k], want[k]) <= 1e-9, k
    dev.close()
