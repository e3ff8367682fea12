"""3D rebuilds whose cells have more candidates near them than the register builder's lanes: it narrows its bands of
squared distance, and the cells that it leaves all the same go to one list of their simulation.  The meshes are the
host tessellator's bit for bit, alone and for two such simulations in one batch."""
import dataclasses

import numpy as np
import pytest

from hydro_rs_amd import fvs, ics
from hydro_rs_amd.mesh import VoronoiMesh

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    if fvs.device_count() < 1:
        pytest.skip("no HIP device")


def _clump(n, share, width, boundary):
    """`share` of n generators uniform in a cube of `width` around the centre, the others in the whole box."""
    rng = np.random.default_rng(n)
    loc = rng.random((n, 3))
    k = int(n * share)
    loc[n - k:] = 0.5 + width * (loc[n - k:] - 0.5)
    cfg = fvs.Config(dim=3, box=(1.0, 1.0, 1.0), gamma=1.4, cfl=0.3, solver=fvs.HLLC, boundary=boundary,
                     motion=fvs.FLUID, t_end=1.0, sync_all=True)
    return ics._finish("clump", cfg, loc, np.ones(n), np.zeros((n, 3)), np.ones(n))


# densities up to some 60 (0.5 in 0.2) and 12 (0.75 in 0.4) times the rest; 64/65 generators
CASES = [(64, 0.5, 0.2), (65, 0.5, 0.2), (257, 0.5, 0.2), (1000, 0.5, 0.2), (2000, 0.75, 0.4)]


@pytest.mark.parametrize("boundary", [fvs.PERIODIC, fvs.REFLECTIVE])
@pytest.mark.parametrize("n, share, width", CASES)
def test_clumped_mesh_equals_host(n, share, width, boundary):
    print(f"[v3 left] n={n} share={share} width={width} boundary={boundary}", flush=True)
    prob = _clump(n, share, width, boundary)
    dev = ics.build_device_sim(prob)
    assert dev.run(1) == 1
    loc = dev.get_state(["loc"])["loc"].reshape(3, n).T.copy()
    want, got = VoronoiMesh(3, prob.cfg.box, boundary == fvs.PERIODIC, loc).as_dict(), dev.get_mesh()
    assert got["n_faces"] == want["n_faces"]
    for k in want:
        if isinstance(want[k], np.ndarray):
            assert np.array_equal(got[k], want[k]), k
    dev.close()


def test_cells_of_many_entries_equal_host():
    """Random generators: one cell in a hundred has more CSR entries than its bucket holds, chained behind it."""
    print("[v3 left] chained entries", flush=True)
    prob = _clump(20000, 0.0, 1.0, fvs.PERIODIC)
    many = prob.mesh.as_dict()["count"] > 24
    assert 0 < many.sum() < prob.n // 20
    dev = ics.build_device_sim(prob)
    assert dev.run(1) == 1
    loc = dev.get_state(["loc"])["loc"].reshape(3, prob.n).T.copy()
    want, got = VoronoiMesh(3, prob.cfg.box, True, loc).as_dict(), dev.get_mesh()
    for k in ("n_faces", "left", "right", "offset", "count", "conn"):
        assert np.array_equal(got[k], want[k]), k
    dev.close()


def test_clumped_batch_members_equal_alone():
    print("[v3 left] batch", flush=True)
    probs = [_clump(1000, 0.5, 0.2, fvs.PERIODIC), ics.sedov_2d(side=16, t_end=0.01),
             _clump(2000, 0.75, 0.4, fvs.REFLECTIVE)]
    probs[2] = dataclasses.replace(probs[2], cfg=dataclasses.replace(probs[2].cfg, sync_all=False))
    batch = fvs.Batch.for_problems(probs, headroom=1.25)
    batch.run(3)
    for s in (0, 2):
        alone = ics.build_device_sim(probs[s])
        assert alone.run(3) == 3
        a, b = batch.get_state(s), alone.get_state()
        for k in b:
            assert np.array_equal(a[k], b[k]), (s, k)
        alone.close()
