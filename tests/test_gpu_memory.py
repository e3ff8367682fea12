"""Device memory of moving meshes: their rebuild's buffers take the place of what only fixed meshes use."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from hydro_rs_amd import _lib, fvs, ics

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    if fvs.device_count() < 1:
        pytest.skip("no HIP device")


def _free():
    free, total = C.c_size_t(0), C.c_size_t(0)
    assert _lib.hfv().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _moving(prob):
    return dataclasses.replace(prob, cfg=dataclasses.replace(prob.cfg, motion=fvs.FLUID))


def test_moving_context_takes_no_more_than_a_fixed_one():
    fixed = ics.kelvin_helmholtz_3d(side=64, t_end=0.1)
    used = []
    for prob in (fixed, fixed, _moving(fixed)):  # (the first one also pays for the runtime's own allocations)
        before = _free()
        sim = ics.build_device_sim(prob)
        used.append((before - _free()) / prob.n)
        sim.close()
    print(f"[memory] bytes a cell: fixed {used[1]:.0f}, moving {used[2]:.0f}", flush=True)
    assert used[2] <= used[1]


def test_rebuild_buffers_of_a_batch():
    """A batch allocates the rebuild's buffers when the first moving mesh comes: a face in provisional order (64 bytes),
    24 entries a cell (192) and seven words a cell; 1 % for the sums and the allocator's granularity."""
    fixed = ics.kelvin_helmholtz_3d(side=48, t_end=0.1)
    cells, faces = 2 * fixed.n, 2 * fixed.mesh.n_faces
    caps = [np.array([v, v], dtype=np.int64) for v in (fixed.n, fixed.mesh.n_faces, fixed.mesh.conn.size)]
    b = fvs.Batch(*caps)
    b.load(0, fixed)
    before = _free()
    b.load(1, _moving(fixed))
    grown, want = before - _free(), 64 * faces + (192 + 28) * cells
    print(f"[memory] rebuild buffers: {grown / cells:.0f} bytes a cell, of which {want / cells:.0f} are named", flush=True)
    assert grown <= 1.01 * want + (9 << 21)
    b.run(2)
    b.close()
