"""CPU check of the device footprint stated for a beamlet call (tests/audit/footprint_check.hip): it counts the
buffers that the call's job holds, the zeros around every REV line and the lines' grids among them."""
import json
import os
import subprocess

import pytest

from endtoend_amd import workloads as W

from tests.shim_case import write_case

CHECK = os.path.join(os.path.dirname(os.path.abspath(__file__)), "audit", "_build", "footprint_check")


@pytest.mark.parametrize("case", ["small", "batched"])
def test_footprint_counts_every_buffer(tmp_path, case):
    w = W.small(n=32, hetero=True) if case == "small" else W.cfg3(nbeams=5)
    write_case(str(tmp_path), w.spec, w.beams, w.fmaps)
    r = subprocess.run([CHECK, str(tmp_path)], capture_output=True, text=True, timeout=300)
    assert r.stdout, r.stderr
    out = json.loads(r.stdout.strip().splitlines()[-1])
    assert out["beams"] == len(w.beams) and out["stated"] == out["held"] > 0, out
    assert r.returncode == 0 and out["differences"] == 0
