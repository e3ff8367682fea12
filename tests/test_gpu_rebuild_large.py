"""Rebuilds on either side of the size from which the chunk sums are scanned by kernels of their own (2048 chunks of
256 cells): the device's mesh is the host tessellator's, indices exactly and areas bit for bit."""
import numpy as np
import pytest

from hydro_rs_amd import fvs, ics
from hydro_rs_amd.mesh import VoronoiMesh

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    if fvs.device_count() < 1:
        pytest.skip("no HIP device")


# 724^2 cells are 2048 chunks, 725^2 are 2054, 1100^2 need five rounds of a scan's 1024 threads
@pytest.mark.parametrize("side", [724, 725, 1100])
def test_large_mesh_equals_host(side):
    print(f"[rebuild large] side={side}", flush=True)
    loc = ics.jittered_grid(2, side, (1.0, 1.0, 1.0), 0.2, np.random.default_rng(side))
    n = loc.shape[0]
    cfg = fvs.Config(dim=2, box=(1.0, 1.0, 1.0), gamma=1.4, cfl=0.3, solver=fvs.HLLC, boundary=fvs.PERIODIC,
                     motion=fvs.FLUID, t_end=1.0, sync_all=True)
    dev = ics.build_device_sim(ics._finish("grid", cfg, loc, np.ones(n), np.full((n, 3), [0.3, 0.1, 0.0]), np.ones(n)))
    assert dev.run(2) == 2
    loc = dev.get_state(["loc"])["loc"].reshape(3, n).T.copy()
    want, got = VoronoiMesh(2, cfg.box, True, loc).as_dict(), dev.get_mesh()
    assert got["n_faces"] == want["n_faces"]
    for k in ("left", "right", "offset", "count", "conn", "area"):
        assert np.array_equal(got[k], want[k]), k
    dev.close()
