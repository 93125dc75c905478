"""CPU check of the cone kernel's segment-sum walk as a wave runs it (tests/audit/joint_walk_check.hip): both
directions of a destination together, lanes that go on after their own end, radial tables that end inside the
line, against the walks' sums in FP64 over the same centres, with every table beside an unmapped page."""
import json
import os
import subprocess

CHECK = os.path.join(os.path.dirname(os.path.abspath(__file__)), "audit", "_build", "joint_walk_check")


def test_joint_walk():
    r = subprocess.run([CHECK, "4000", "5"], capture_output=True, text=True, timeout=300)
    assert r.stdout, f"ended with {r.returncode}"
    out = json.loads(r.stdout.strip().splitlines()[-1])
    assert r.returncode == 0 and out["mismatch"] == 0, out
    assert out["destinations"] > 200000 and out["late_lanes"] > 100000
    assert out["lines_beyond_the_radii"] > 1000 and out["single_cell_lines"] > 50
