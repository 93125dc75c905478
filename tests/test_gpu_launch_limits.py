"""Calls whose kernels take more workgroups than one launch holds (2^24 - 1 of 256 threads): they run in
several launches, and every part of the result is what a smaller call gives, bit for bit."""
import numpy as np
import pytest

from endtoend_amd import engine as E
from endtoend_amd import workloads as W
from endtoend_amd.engine import Engine

pytestmark = pytest.mark.gpu


def test_columns_of_many_small_boxes_and_a_huge_one():
    """One beamlet whose box spans a wide, flat grid beside 400 with narrow boxes: the column passes' chunks of
    rows (those of the largest box for every beamlet) exceed one launch."""
    n = 3300
    ph = W.Phantom(np.full((4, n, n), 0.02, np.float32), 0.1)
    spec = W.problem(ph, nphi=2, ntheta=4, spacing=0.5, kernel_extent=0.3, max_rev_size=(1024, 1024, 1024))
    beams = [E.make_beam(45.0, 0.0, 0.0, sad=400.0, fmap_size=(1, 1), beamlet_size=(0.5, 0.5)),
             E.make_beam(0.0, 0.0, 0.0, sad=400.0, fmap_size=(400, 1), beamlet_size=(0.5, 0.5))]
    fmaps = [np.ones((1, 1), np.float32), np.ones((1, 400), np.float32)]
    with Engine(spec) as eng:
        eng.set_schedule("bl_streams", 1)  # (both beams then fit into one job)
        print("[case] both beams", flush=True)
        both = eng.beamlet_dose(beams, fmaps, threshold=1e-4)
        print("[case] each beam alone", flush=True)
        alone = [eng.beamlet_dose([b], [f], threshold=1e-4) for b, f in zip(beams, fmaps)]
    rows = np.unique(both[0][2] // np.uint64(n) % np.uint64(n)).size
    assert rows > 1500  # the diagonal beamlet's column reaches far over the grid
    one = [(i, c[1], c[2], c[3]) for i, cols in enumerate(alone) for c in cols]
    assert len(both) == len(one) == 401
    for x, y in zip(both, one):
        assert x[:2] == y[:2]
        assert np.array_equal(x[2], y[2]) and np.array_equal(x[3].view(np.uint32), y[3].view(np.uint32))


def test_terma_of_a_thin_box():
    """A calc_bbox one voxel thick along x fills a sixteenth of its workgroups' lanes."""
    ny, nz = 16384, 16400
    spec = W.problem(W.Phantom(np.ones((nz, ny, 1), np.float32), 0.01), nphi=2, ntheta=4, max_rev_size=(800, 800, 800))
    beam = E.make_beam(0.0, 0.0, 0.0, iso=(0.0, 0.0, 0.0), sad=100.0, fmap_size=(3, 3), beamlet_size=(0.3, 0.3))
    fmap = np.arange(1.0, 10.0, dtype=np.float32).reshape(3, 3)
    with Engine(spec) as eng:
        print("[case] whole box", flush=True)
        whole = eng.beam_terma(beam, fmap)
    z = np.nonzero(whole.any(axis=(1, 2)))[0]
    assert z.size > 50
    lo = int(z[0]) - 8
    spec.bbox_start, spec.bbox_size = (0, 0, lo), (1, ny, int(z[-1]) + 8 - lo)
    with Engine(spec) as eng:
        print("[case] field only", flush=True)
        part = eng.beam_terma(beam, fmap)
    np.testing.assert_array_equal(whole[lo:lo + part.shape[0]].view(np.uint32), part.view(np.uint32))
    assert not whole[:lo].any() and not whole[lo + part.shape[0]:].any()


def test_projection_of_half_a_billion_beamlets():
    n, m = 8, 8000
    spec = W.problem(W.water_cube(16, 1.0), nphi=2, ntheta=4)
    mask = np.zeros((16, 16, 16), np.uint8)
    mask[4:11, 6:9, 5:12] = 1
    beams = [E.make_beam(40.0 * i, 10.0 * i, 0.0, fmap_size=(m, m), beamlet_size=(0.002, 0.002)) for i in range(n)]
    with Engine(spec) as eng:
        print("[case] all beams", flush=True)
        got = eng.fluence_projection(mask, beams)
        for i in (0, n - 1):
            print(f"[case] beam {i}", flush=True)
            one = eng.fluence_projection(mask, [beams[i]])[0]
            np.testing.assert_array_equal(got[i], one)
            assert 0 < int(one.sum()) < m * m
