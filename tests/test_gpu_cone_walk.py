"""The cone kernel's segment-sum walk and line resample where they can go wrong, against the CPU oracle
(the repository's dose bars) and against the sequential walk of the same build (lines that end inside
the radial table may lose or gain their last sample to FP32 rounding: the dose bar): grids of a
few voxels (no interior samples), lines parallel to the grid, a calc_bbox off the grid's faces,
vacuum at both ends of the lines, and radial tables that end inside the lines (the walk's exits)."""
import numpy as np
import pytest

from endtoend_amd import workloads as W
from endtoend_amd.engine import Engine
from oracle import oracle as O
from tests.dose_metrics import gamma_pass_rate, max_err_pct

pytestmark = pytest.mark.gpu

DOSE_TOL_PCT = 0.5
GAMMA_MIN = 0.995

CASES = {
    "tiny-6": dict(n=6, voxel=1.0, gantry=20.0, couch=10.0, fmap=(4, 4), beamlet=(1.0, 1.0)),
    "tiny-11": dict(n=11, voxel=0.7, gantry=75.0, couch=-30.0, fmap=(5, 5), beamlet=(1.0, 1.0)),
    "parallel-g90": dict(n=26, voxel=0.5, gantry=90.0, hetero=True),
    "bbox-g17": dict(n=30, voxel=0.5, gantry=17.0, couch=8.0, hetero=True, bbox=((5, 3, 1), (21, 25, 28))),
    "vacuum-g40": dict(n=34, voxel=0.5, gantry=40.0, couch=25.0, hetero=True),
    "exits-g33": dict(n=34, voxel=0.5, gantry=33.0, couch=12.0, hetero=True),
    "exits-short-g140": dict(n=30, voxel=0.5, gantry=140.0, couch=-50.0),
}


@pytest.mark.parametrize("name", list(CASES))
def test_cone_walk_edges(name):
    w = W.small(**CASES[name])
    rng = np.random.default_rng(3)
    w.spec.density *= (1.0 + 0.02 * rng.standard_normal(w.spec.density.shape)).astype(np.float32)
    if name.startswith("vacuum"):
        w.spec.density[:, :5, :] = 0.0
        w.spec.density[:, -5:, :] = 0.0
        w.spec.density[:, :, :4] = 0.0
    if name.startswith("exits"):
        w.spec.radii = (w.spec.radii * np.float32(0.0371 if "short" in name else 0.1337)).astype(np.float32)
    print(f"[case] {name}", flush=True)
    with Engine(w.spec) as eng:
        eng.set_schedule("cone_ramp_min", 1 << 20)
        seq = eng.beam_dose(w.beams, w.fmaps)
        eng.set_schedule("cone_ramp_min", 1)
        ramp = eng.beam_dose(w.beams, w.fmaps)
    d, _ = O.beam_dose(w.spec, w.beams, w.fmaps)
    assert d.max() > 0
    for got in (seq, ramp):
        assert max_err_pct(d, got) <= DOSE_TOL_PCT
        assert gamma_pass_rate(d, got, voxel_mm=10 * w.spec.voxel[0]) >= GAMMA_MIN
    assert max_err_pct(seq, ramp) <= DOSE_TOL_PCT
    np.testing.assert_array_equal(ramp != 0, seq != 0)
