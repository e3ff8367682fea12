"""The register builders of the 2D and 3D rebuilds at the sizes where they hand a cell on: every mesh is the host
tessellator's, bit for bit."""
import numpy as np
import pytest

from hydro_rs_amd import fvs, ics
from hydro_rs_amd.mesh import VoronoiMesh
from tests.helpers import star_problem

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    if fvs.device_count() < 1:
        pytest.skip("no HIP device")


def _problem(dim, loc, boundary):
    loc = np.hstack([loc, np.zeros((len(loc), 3 - loc.shape[1]))])
    n = len(loc)
    cfg = fvs.Config(dim=dim, box=(1.0, 1.0, 1.0), gamma=1.4, cfl=0.3, solver=fvs.HLLC, boundary=boundary,
                     motion=fvs.FLUID, t_end=1.0, sync_all=True)
    return ics._finish("limits", cfg, loc, np.ones(n), np.zeros((n, 3)), np.ones(n))


def _assert_host_mesh(prob):
    dev = ics.build_device_sim(prob)
    assert dev.run(1) == 1
    loc = dev.get_state(["loc"])["loc"].reshape(3, prob.n).T.copy()
    want = VoronoiMesh(prob.cfg.dim, prob.cfg.box, prob.cfg.boundary == fvs.PERIODIC, loc).as_dict()
    got = dev.get_mesh()
    assert got["n_faces"] == want["n_faces"]
    for k in want:
        if isinstance(want[k], np.ndarray):
            assert np.array_equal(got[k], want[k]), k
    dev.close()


# a 2D cell has its edges on 16 lanes
@pytest.mark.parametrize("ring", [14, 15, 16, 17, 18])
@pytest.mark.parametrize("boundary", [fvs.PERIODIC, fvs.REFLECTIVE])
def test_2d_cell_edges(ring, boundary):
    print(f"[limits] 2D ring {ring} boundary {boundary}", flush=True)
    base = _problem(2, np.random.default_rng(1).random((9, 2)), fvs.PERIODIC)
    prob = star_problem(base, ring, boundary)
    assert prob.mesh.as_dict()["count"][0] == ring
    _assert_host_mesh(prob)


# a 2D cell ranks 96 candidates: n - 1 of them around the middle generator, whose 5 x 5 bins hold all of them
@pytest.mark.parametrize("n", [95, 96, 97, 98, 99])
def test_2d_candidates(n):
    print(f"[limits] 2D candidates {n - 1}", flush=True)
    loc = np.random.default_rng(n).uniform(0.3, 0.7, (n, 2))
    loc[0] = 0.5
    nb = int(np.sqrt(n))
    assert np.all(np.abs(np.floor(loc * nb) - np.floor(0.5 * nb)) <= 2)
    _assert_host_mesh(_problem(2, loc, fvs.REFLECTIVE))


# a 3D cell has its vertices on 64 lanes: `ring` faces are 2 ring - 4 of them, more while it is clipped
@pytest.mark.parametrize("ring", [28, 30, 32, 33, 34, 35, 36])
@pytest.mark.parametrize("boundary", [fvs.PERIODIC, fvs.REFLECTIVE])
def test_3d_cell_vertices(ring, boundary):
    print(f"[limits] 3D ring {ring} boundary {boundary}", flush=True)
    base = _problem(3, np.random.default_rng(1).random((27, 3)), fvs.PERIODIC)
    prob = star_problem(base, ring, boundary)
    assert prob.mesh.as_dict()["count"][0] == ring
    _assert_host_mesh(prob)


# a face of 12 vertices fits a lane's registers: two generators with k others around the middle of their axis
@pytest.mark.parametrize("k", [11, 12, 13, 14])
def test_3d_face_vertices(k):
    print(f"[limits] 3D face of {k} vertices", flush=True)
    rng = np.random.default_rng(k)
    g = (np.arange(5) + 0.5) / 5
    grid = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3) + rng.uniform(-0.02, 0.02, (125, 3))
    c = np.full(3, 0.5)
    a = 2 * np.pi * (np.arange(k) + 0.25) / k
    ring = c + 0.12 * np.stack([np.cos(a), np.sin(a), rng.uniform(-1e-3, 1e-3, k)], -1)
    ends = c + np.array([[0, 0, -0.05], [0, 0, 0.05]])
    prob = _problem(3, np.concatenate([ends, ring, grid[np.linalg.norm(grid - c, axis=1) > 0.2]]), fvs.PERIODIC)
    m = prob.mesh.as_dict()
    mine = m["conn"][m["offset"][0]: m["offset"][0] + m["count"][0]]
    others = set(m["left"][mine]) | set(m["right"][mine])
    assert set(range(k + 2)) <= others  # the face between the two touches a face with each of the ring
    _assert_host_mesh(prob)


# the first band of a 3D cell ranks 64 candidates: n - 1 of them within it for every generator
@pytest.mark.parametrize("n", [63, 64, 65, 66, 67, 80])
def test_3d_candidates(n):
    print(f"[limits] 3D candidates {n - 1}", flush=True)
    loc = np.random.default_rng(n).uniform(0.3, 0.7, (n, 3))
    _assert_host_mesh(_problem(3, loc, fvs.REFLECTIVE))
