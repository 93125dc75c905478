"""GPU TERMA over calc_bbox sizes around its 16x4x4 workgroups and beams along every axis from both ends
(each has its own order of the planes), against the oracle: the same voxels are non-zero, values
within the tolerance of the TERMA parity test (FP32 rounding of the fetch coordinates)."""
import numpy as np
import pytest

from endtoend_amd import workloads as W
from endtoend_amd.engine import Engine
from oracle import oracle as O

pytestmark = pytest.mark.gpu

BOXES = {
    "one voxel": ((20, 20, 20), (1, 1, 1)),
    "one workgroup": ((12, 18, 18), (16, 4, 4)),
    "one over": ((11, 17, 18), (17, 5, 5)),
    "flat": ((2, 19, 3), (37, 2, 33)),
    "eight rows": ((1, 2, 3), (31, 32, 35)),
    "ragged": ((3, 1, 0), (35, 39, 40)),
}


@pytest.mark.parametrize("gantry,couch", [(0.0, 0.0), (180.0, 0.0), (90.0, 0.0), (270.0, 0.0), (90.0, 88.0),
                                          (270.0, 80.0), (37.0, 11.0)])
@pytest.mark.parametrize("box", list(BOXES))
def test_terma_shapes(box, gantry, couch):
    w = W.small(n=40, voxel=0.5, gantry=gantry, couch=couch, hetero=True, fmap=(9, 7), beamlet=(1.0, 1.1),
                bbox=BOXES[box])
    print(f"[case] {box} gantry {gantry} couch {couch}", flush=True)
    with Engine(w.spec) as eng:
        got = eng.beam_terma(w.beams[0], w.fmaps[0])
    ref, _ = O.terma(w.spec, w.beams[0], w.fmaps[0])
    assert np.count_nonzero(ref) > 0
    np.testing.assert_array_equal(got != 0, ref != 0)
    np.testing.assert_allclose(got, ref, rtol=2e-5, atol=1e-7 * float(ref.max()))
