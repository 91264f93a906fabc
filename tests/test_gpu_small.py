"""The l x l kernels (small.hip) and the block-diagonal product at the edges of their tilings: l at
and around the multiples of 16, row counts at and around 64 and 256, spectra that the one-sided
Jacobi takes and ones whose Cholesky pivots send it back to the two-sided form."""
import numpy as np
import pytest

import mcnla_amd as mc
import oracle

pytestmark = pytest.mark.gpu

EDGES = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64]


def params(m, n, l, N):
    return mc.Parameters().setSize(m, n).setRank(l).setOverRank(0).setNumSketch(N)


def basis(rng, m, l):
    return np.linalg.qr(rng.standard_normal((m, l)))[0]


def graded(rng, m, l, decades):
    """(m x l, its singular values): 1 down to 10^-decades, random singular vectors."""
    s = np.logspace(0, -decades, l)
    return (basis(rng, m, l) * s) @ basis(rng, l, l).T, s


@pytest.mark.parametrize("l,m", list(zip(EDGES, [63, 64, 65, 255, 256, 257, 300, 511, 513, 127, 300,
                                                 129, 260])))
@pytest.mark.parametrize("precision", [mc.PREC_F64, mc.PREC_MIXED_BF16])
def test_orthogonalizer_edges(l, m, precision):
    """Q = Y V diag(w)^-1/2 of Y with singular values 1 .. 1e-2, a different scale per sketch.  The
    Gram matrix's rounding (l eps) over its smallest gap (0.13 of 1e-4 at l = 64) bounds the FP64
    columns by 1e-9 l / 64 or so; a mixed collection rounds Q to FP32 (6e-8)."""
    rng = np.random.default_rng(100 * l + m)
    N = 3
    Y = np.hstack([graded(rng, m, l, 2)[0] * sc for sc in (1.0, 3e5, 1e-7)])
    if precision != mc.PREC_F64:
        Y = Y.astype(np.float32)
    o = mc.GramianOrthogonalizer(params(m, m, l, N), precision=precision)
    Q = mc.DeviceArray.from_numpy(np.ascontiguousarray(Y))
    o(Q)
    q = Q.numpy().astype(np.float64)
    ref, bad = oracle.gramian_orthogonalize(Y.astype(np.float64), l, N)
    assert bad == 0
    sign = np.sign(np.sum(q * ref, axis=0))
    assert np.abs(q * sign - ref).max() < (1e-8 if precision == mc.PREC_F64 else 2e-7)


@pytest.mark.parametrize("l", EDGES)
@pytest.mark.parametrize("decades", [6, 8])
def test_former_edges(l, decades):
    """Singular values 1 .. 10^-decades: sigma_j = ||Z w_j|| with w_j from the Gram matrix, whose
    rounding tilts w_j towards the larger ones by about eps / sigma_j.  At 1e-6 the pivots pass; LAPACK's
    eigensolver leaves 6.4e-10 there at l = 64, six times that is allowed.  At 1e-8 the smallest
    eigenvalues drown in rounding and the pivots fail: only the leading half (1e-4) is compared."""
    rng = np.random.default_rng(l)
    m, n = 300, 200
    W, s = graded(rng, n, l, decades)
    Q = basis(rng, m, l)
    f = mc.SvdFormer(params(m, n, l, 1), True)
    f(mc.DeviceArray.from_numpy(np.asfortranarray(Q @ W.T)), mc.DeviceArray.from_numpy(Q))
    S, U = f.vectorS(), f.matrixU()
    keep = l if decades == 6 else (l + 1) // 2
    err = np.abs(S - s) / s
    assert np.max(err[:keep]) < (4e-9 if decades == 6 else 2e-8)
    assert np.abs(U.T @ U - np.eye(l)).max() < 1e-12


@pytest.mark.parametrize("k,p,N", [(1, 0, 3), (8, 7, 3), (10, 6, 3), (10, 7, 2), (20, 11, 3),
                                   (20, 12, 2), (20, 13, 2), (30, 17, 2), (30, 18, 2), (30, 19, 2),
                                   (50, 13, 2), (50, 14, 3)])
def test_solve_edges(k, p, N):
    """The Cholesky route of a solve against the oracle's eigen transforms."""
    m, n, l = 400, 150, k + p
    rng = np.random.default_rng(l)
    A = (basis(rng, m, n) * 0.9 ** np.arange(n)) @ basis(rng, n, n).T
    om = oracle.omega_ref(3, n, N * l, col_block=True)
    Q, _ = oracle.gramian_orthogonalize(oracle.sketch(A, om), l, N)
    Qb, iters = oracle.kn_rowblock(Q, l, N, 256, 1e-4)
    S, U, _ = oracle.svd_former(A, Qb, k)
    P = mc.Parameters().setSize(m, n).setRank(k).setOverRank(p).setNumSketch(N)
    s = mc.Solver(P, seed=3, omega_mode=mc.OMEGA_REFERENCE)
    s.solve(mc.DeviceArray.from_numpy(np.asfortranarray(A)))
    assert abs(s.iteration() - iters) <= 1
    assert np.max(np.abs(s.vectorS() - S) / S) < 1e-9
    assert np.abs(U @ U.T - s.matrixU() @ s.matrixU().T).max() < 1e-8


def test_solve_many_sketches():
    """N = 4200 sketches of one column: 8.8 million block pairs in the congruence B_s = T'GT, more
    workgroups of 512 than one grid dimension holds."""
    m, n, N = 60, 40, 4200
    rng = np.random.default_rng(8)
    A = (basis(rng, m, n) * 0.7 ** np.arange(n)) @ basis(rng, n, n).T
    om = oracle.omega_ref(3, n, N, col_block=True)
    Q, _ = oracle.gramian_orthogonalize(oracle.sketch(A, om), 1, N)
    Qb, iters = oracle.kn_rowblock(Q, 1, N, 256, 1e-4)
    S, U, _ = oracle.svd_former(A, Qb, 1)
    P = mc.Parameters().setSize(m, n).setRank(1).setOverRank(0).setNumSketch(N)
    s = mc.Solver(P, seed=3, omega_mode=mc.OMEGA_REFERENCE, route=mc._lib.ROUTE_SKETCH)
    s.solve(mc.DeviceArray.from_numpy(np.asfortranarray(A)))
    assert abs(s.iteration() - iters) <= 1
    assert np.max(np.abs(s.vectorS() - S) / S) < 1e-9
    assert np.abs(U @ U.T - s.matrixU() @ s.matrixU().T).max() < 1e-8
