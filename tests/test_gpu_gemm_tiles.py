"""The FP64 products' register-fed tiles (gemm_f64.hip, 32 x 32 and 64 x 64) at the edges of their
tilings, through the sketch Y = A Omega: rows and columns at and around multiples of 32, K at and
around the 16-wide stages (fewer of them than waves too), both orders, FP32 and FP64, a leading
dimension that no 16-byte load could take.  Tolerance: the dot products' rounding, K eps |A||Omega|
entry by entry."""
import numpy as np
import pytest

import mcnla_amd as mc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", ["F", "C"])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m,n,l,N", [
    (31, 15, 1, 1), (32, 16, 2, 16), (33, 17, 3, 11), (64, 127, 8, 8), (65, 128, 13, 5),
    (95, 129, 31, 1), (129, 143, 32, 3), (257, 1, 1, 7), (1000, 333, 20, 4),
    (4001, 777, 17, 31), (9001, 130, 33, 20),   # 64 x 64 tiles in several rounds
    (2000, 1000, 20, 8), (256, 64, 32, 4),      # sizes the DMA tiles could take
])
def test_sketch_tiles(m, n, l, N, dtype, order):
    rng = np.random.default_rng(m + n)
    A = np.asarray(rng.standard_normal((m, n)), dtype=dtype, order=order)
    P = mc.Parameters().setSize(m, n).setRank(l).setOverRank(0).setNumSketch(N)
    s = mc.ColBlockGaussianProjectionSketcher(P, seed=7)
    Q = P.createCollectionQ()
    s(mc.DeviceArray.from_numpy(A), Q)
    om = s.omega()
    a = A.astype(np.float64)
    bound = 2.0 * (n + 8) * np.finfo(np.float64).eps * (np.abs(a) @ np.abs(om))
    assert np.all(np.abs(Q.numpy() - a @ om) <= bound)
