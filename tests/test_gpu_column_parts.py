"""Beamlet columns large enough to reach the sink in several parts, and small ones beside them: every
column's keys and values are those of its dense column (the same arithmetic, so bit for bit), in request
order, with one beam, with two, and with a call of one beamlet."""
import numpy as np
import pytest

from endtoend_amd import workloads as W
from endtoend_amd.engine import Engine, make_beam
from oracle import oracle as O

pytestmark = pytest.mark.gpu

PART = 1 << 18  # entries a part of the columns is worth


@pytest.fixture(scope="module")
def eng():
    w = W.small(n=64, voxel=0.25, hetero=True)
    w.spec.kernel_extent = 1.0
    e = Engine(w.spec)
    yield w, e
    e.close()


@pytest.mark.parametrize("maps", [((14, 14),), ((14, 14), (10, 12)), ((1, 1),), ((3, 2), (14, 14))])
def test_columns_in_parts(eng, maps):
    w, e = eng
    thr = 1e-4
    print(f"[case] maps {maps}", flush=True)
    beams = [make_beam(20.0 + 65.0 * i, 10.0 * i, 0.0, fmap_size=m, beamlet_size=(0.5, 0.5)) for i, m in enumerate(maps)]
    fmaps = [np.ones((m[1], m[0]), np.float32) for m in maps]
    cols = e.beamlet_dose(beams, fmaps, threshold=thr)
    assert [(c[0], c[1]) for c in cols] == [(i, k) for i, m in enumerate(maps) for k in range(m[0] * m[1])]
    total = 0
    q = 0
    for b, f in zip(beams, fmaps):
        for d in e.beamlet_dense(b, f):
            ek, ev, _, _ = O.sparsify(d, w.spec.size, w.spec.bbox_start, w.spec.bbox_size, thr)
            k, v = cols[q][2], cols[q][3]
            assert np.array_equal(k, ek), f"column {q}"
            assert np.array_equal(v.view(np.uint32), ev.view(np.uint32)), f"column {q}"
            total += k.size
            q += 1
    if maps != ((1, 1),):
        assert total > 2 * PART
