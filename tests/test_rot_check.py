"""CPU check of the geometry's short forms (tests/audit/rot_check.hip): rotations about known axes
against the general Rodrigues form, quotients from a stored reciprocal against the division, 24-bit
multiply-adds against the plain product; no difference may occur."""
import json
import os
import subprocess

CHECK = os.path.join(os.path.dirname(os.path.abspath(__file__)), "audit", "_build", "rot_check")


def test_short_forms_equal_the_general_ones():
    r = subprocess.run([CHECK, "1000000", "3"], capture_output=True, text=True, timeout=300)
    out = json.loads(r.stdout.strip().splitlines()[-1])
    assert r.returncode == 0, out
    assert out["rotations"] == 4000000 and out["divisions"] == 1000000
    assert out["rotation_differences"] == out["division_differences"] == out["mad24_differences"] == 0
