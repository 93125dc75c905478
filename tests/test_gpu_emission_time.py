"""The emission of a job's columns costs the device the same whether they stay there or go to a sink in parts: its
time is the longest row's serial chain, so an emission split over the parts would cost it once for each."""
import pytest

from endtoend_amd import workloads as W
from endtoend_amd.engine import Engine

pytestmark = pytest.mark.gpu


def test_parts_do_not_multiply_the_emission():
    w = W.cfg3(nbeams=1)
    best = {}
    with Engine(w.spec) as eng:
        eng.set_schedule("bl_streams", 1)
        for keep in (None, False) * 4:
            print(f"[case] keep {keep}", flush=True)
            eng.profile(True)
            eng.profile_reset()
            eng.beamlet_dose(w.beams, w.fmaps, threshold=1e-4, keep=keep)
            eng.sync()
            ms = eng.profile_read()["bl_compact"]["ms"]
            best[keep] = min(ms, best.get(keep, ms))
    assert best[False] < 2.0 * best[None], best
