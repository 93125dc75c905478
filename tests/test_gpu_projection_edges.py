"""GPU structure projection at the edges of its kernels: masks at the grid's corners, in one voxel, empty
and full, grids whose voxel count is no multiple of four, and beamlet counts below and between multiples
of 64.  The maps are decisions, so they must equal the oracle's."""
import numpy as np
import pytest

from endtoend_amd import engine as E
from endtoend_amd import workloads as W
from endtoend_amd.engine import Engine
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _mask(kind, shape):
    m = np.zeros(shape, np.uint8)
    if kind == "first":
        m[0, 0, 0] = 1
    elif kind == "last":
        m[-1, -1, -1] = 255
    elif kind == "two":
        m[1, 2, 3] = 1
        m[-2, -1, -3] = 7
    elif kind == "full":
        m[:] = 1
    elif kind == "slab":
        m[:, shape[1] // 2, :] = 1
    return m


@pytest.mark.parametrize("n", [(7, 9, 11), (16, 16, 16), (33, 20, 5)])
@pytest.mark.parametrize("kind", ["first", "last", "two", "full", "slab", "empty"])
def test_projection_edges(n, kind):
    ph = W.thorax(n[0], n[1], n[2], 0.5)
    spec = W.problem(ph, nphi=4, ntheta=4, max_rev_size=(800, 800, 800))
    mask = _mask(kind, (n[2], n[1], n[0]))
    beams = [E.make_beam(g, c, coll, iso=(0.1, 0.0, -0.2), fmap_size=(fx, fy), beamlet_size=(0.7, 0.6))
             for g, c, coll, fx, fy in ((0.0, 0.0, 0.0, 1, 1), (41.0, 12.0, 5.0, 9, 7), (90.0, 0.0, 0.0, 13, 5),
                                        (180.0, 35.0, 0.0, 8, 8), (270.0, -60.0, 30.0, 3, 21))]
    print(f"[case] {n} {kind}", flush=True)
    with Engine(spec) as eng:
        got = eng.fluence_projection(mask, beams)
    ref = O.fluence_projection(spec, mask, beams)
    for g, r in zip(got, ref):
        assert np.array_equal(g, r)
    if kind == "empty":
        assert all(not g.any() for g in got)
    if kind == "full":
        assert sum(float(r.sum()) for r in ref) > 20
