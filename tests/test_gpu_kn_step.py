"""The Kolmogorov-Nagumo iteration's kernels (integrate.hip) at the edges of their tilings: l at and
around the multiples of 16, Nl at and past the workgroup and partial-sum limits (8 x 16 rows, 4096
rows), odd Nl, and sketches from nearly equal (the series form of the l x l step) to nearly
unrelated (the square-root iterations).  Against the oracle, element-wise 1e-8 as for the fixtures."""
import numpy as np
import pytest

import mcnla_amd as mc
import oracle

pytestmark = pytest.mark.gpu


def sketches(m, l, N, spread, seed):
    """N orthonormal m x l bases around one subspace, side by side."""
    rng = np.random.default_rng(seed)
    U, _ = np.linalg.qr(rng.standard_normal((m, l)))
    out = []
    for _ in range(N):
        R, _ = np.linalg.qr(rng.standard_normal((l, l)))
        Q, _ = np.linalg.qr(U @ R + spread / np.sqrt(m) * rng.standard_normal((m, l)))
        out.append(Q)
    return np.ascontiguousarray(np.hstack(out))


@pytest.mark.parametrize("m,l,N,spread", [
    (90, 1, 40, 0.5), (120, 7, 3, 0.5), (150, 15, 5, 1.0), (150, 16, 8, 0.3), (150, 17, 8, 0.3),
    (200, 16, 9, 3.0), (200, 31, 5, 0.05), (200, 32, 4, 2.0), (200, 33, 5, 0.5), (200, 47, 3, 0.5),
    (200, 48, 4, 0.1), (200, 49, 7, 1.0), (200, 63, 2, 0.5), (200, 64, 2, 0.5), (300, 64, 5, 2.0),
    (150, 31, 133, 0.5),  # Nl = 4123: 32-row workgroups, scalar loads
    (150, 64, 65, 0.5),   # Nl = 4160: 32-row workgroups, 16-byte loads
])
def test_kn_iteration_edges(m, l, N, spread):
    Qs = sketches(m, l, N, spread, seed=m + l + N)
    P = mc.Parameters().setSize(m, m).setRank(l).setOverRank(0).setNumSketch(N)
    it = mc.RowBlockKolmogorovNagumoIntegrator(P, 256, 1e-4)
    Qbar = P.createMatrixQbar()
    it(mc.DeviceArray.from_numpy(Qs), Qbar)
    ref, iters = oracle.kn_rowblock(Qs, l, N, 256, 1e-4)
    assert it.iteration() == iters
    assert np.max(np.abs(Qbar.numpy() - ref)) < 1e-8


@pytest.mark.parametrize("l,N", [
    (64, 20),   # Nl = 1280: the columns of a row block in two parts
    (17, 130),  # Nl = 2210, uncut again
    (37, 40),   # Nl = 1480
    (49, 45),   # Nl = 2205, odd
    (33, 128),  # Nl = 4224: 32-row workgroups
    (20, 7),    # Nl = 140: the smallest in two parts
])
def test_kn_product_parts(l, N):
    """The rule that cuts a product's row blocks by columns, on both sides of its lines."""
    Qs = sketches(150, l, N, 0.5, seed=l + N)
    P = mc.Parameters().setSize(150, 150).setRank(l).setOverRank(0).setNumSketch(N)
    it = mc.RowBlockKolmogorovNagumoIntegrator(P, 256, 1e-4)
    Qbar = P.createMatrixQbar()
    it(mc.DeviceArray.from_numpy(Qs), Qbar)
    ref, iters = oracle.kn_rowblock(Qs, l, N, 256, 1e-4)
    assert it.iteration() == iters
    assert np.max(np.abs(Qbar.numpy() - ref)) < 1e-8
