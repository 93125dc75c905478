"""GPU fluence-map convolution at every kernel width (each has its own unrolled row) and at map sizes
around the tile of 16: bit-identical to the oracle, the same FP32 terms added in the same order."""
import numpy as np
import pytest

from endtoend_amd import workloads as W
from endtoend_amd.engine import Engine
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = Engine(W.small(n=16).spec)
    yield e
    e.close()


@pytest.mark.parametrize("kw", range(1, 32, 2))
def test_convolve_every_kernel_width(eng, kw):
    rng = np.random.default_rng(kw)
    for n, h, w, kh in ((2, 15, 17, 3), (1, 33, 16, 31)):
        print(f"[case] conv n{n} {h}x{w} k{kh}x{kw}", flush=True)
        f = rng.uniform(0, 1, (n, h, w)).astype(np.float32)
        k = rng.uniform(-0.2, 1, (kh, kw)).astype(np.float32)
        got = eng.fluence_convolve(f, k)
        ref = O.fluence_convolve(f, k)
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
