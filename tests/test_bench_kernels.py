"""The kernels whose profiled traffic bench.py looks up exist under the names it uses, and a profile of other kernels
than the present ones is not reported as theirs."""
import json
import shutil
import subprocess

import pytest

import bench
from hydro_rs_amd import _lib, fvs


@pytest.mark.skipif(shutil.which("nm") is None, reason="no nm")
def test_slot_kernels_are_in_the_library():
    out = subprocess.run(["nm", "-C", _lib.HFV_SO], capture_output=True, text=True, check=True).stdout
    have = {ln.split(" ", 2)[2] for ln in out.splitlines() if " hfv::" in ln or " void hfv::" in ln}
    tunings = [None, [{"static_grad": 0}, {"static_grad": 1}]]
    want = {k for slot in bench.ALGO for fp32 in (False, True) for solver in (fvs.EXACT, fvs.HLLC, fvs.AIRS)
            for tuning in tunings for fpt in (1, 2, 4) for k in bench.slot_kernels(slot, fp32, solver, tuning, fpt)}
    assert len(want) > 20
    assert not want - have, sorted(want - have)


def test_traffic_of_other_kernels_is_not_reported(tmp_path, monkeypatch):
    monkeypatch.setattr(bench, "PROFILES", str(tmp_path))
    rec = {"label": "x", "kernels": {"hfv::k": {"traffic_bytes": 7.0}}}
    for kid, want in ((bench.kernels_id(), 7.0), ("0" * 16, None), (None, None)):
        doc = dict(rec, **({"kernels_id": kid} if kid else {}))
        (tmp_path / "x_pmc.md").write_text("TRAFFIC_JSON " + json.dumps(doc) + "\n")
        assert bench.traffic_for("x", "hfv::k") == want
