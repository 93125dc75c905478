"""CPU replay of the beamlet sample stage (tests/audit/sample_replay.hip): the library's own planning builds the
job tables of a workload, the REV store is laid out as the interval and sample kernels do, and the sample
kernel's passes run on the host with the kernel's own functions for the groups of 64 lines that a wave takes.
Every index stays inside its array, the offsets equal a running sum over the lines, the cull keeps every
footprint sample, no sample outside the exact list takes dose, and no line queues more TERMA requests than it
reserves.  On the 50-beam batched workload (every 41st group of every direction), on two beams of the 4pi
precompute (2.5 mm beamlets, 96 cones, every 17th group), on a small heterogeneous grid, and on a batch of more pillars than
the stage tracks."""
import json
import os
import subprocess

import numpy as np
import pytest

from endtoend_amd import engine as E
from endtoend_amd import workloads as W

from tests.shim_case import write_case

REPLAY = os.path.join(os.path.dirname(os.path.abspath(__file__)), "audit", "_build", "sample_replay")


def _many_pillars():
    spec = W.problem(W.water_cube(16, 0.5), nphi=2, ntheta=4, kernel_extent=0.3, max_rev_size=(1024, 1024, 1024))
    beam = E.make_beam(20.0, 15.0, 0.0, fmap_size=(65, 65), beamlet_size=(0.05, 0.05))
    return W.Workload("many pillars", spec, [beam], [np.ones((65, 65), np.float32)])


@pytest.mark.parametrize("case,stride", [("batched", 41), ("4pi", 17), ("small", 1), ("many pillars", 1)])
def test_replay(tmp_path, case, stride):
    w = {"batched": W.cfg3, "4pi": lambda: W.cfg5(indices=[0, 581]),
         "small": lambda: W.small(n=32, gantry=48.0, couch=12.0, hetero=True), "many pillars": _many_pillars}[case]()
    write_case(str(tmp_path), w.spec, w.beams, w.fmaps)
    r = subprocess.run([REPLAY, str(tmp_path), str(stride)], capture_output=True, text=True, timeout=600)
    assert r.stdout, r.stderr
    out = json.loads(r.stdout.strip().splitlines()[-1])
    assert r.returncode == 0 and out["violations"] == 0, out
    assert out["footprint_lines"] > 100 and out["cull_checked"] > 1000 and out["shared_lists"] > 50
    assert out["shortfall"] == 0 and out["max_list"] <= 1024
    assert out["zeros"] == (case != "batched")  # (as one job, its stores are beyond the zeros' 2^30 samples)
    if case == "many pillars":
        assert out["untracked_lines"] == out["footprint_lines"] and out["batches"] == 1
    else:
        assert out["untracked_lines"] == 0 and out["walls_checked"] > 1000
