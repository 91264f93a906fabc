"""FP64 products by residues on the INT8 matrix cores (gemm_residue.hip): the sketch against
extended precision, and the solver's Gram matrices against the FP64 kernels, at sizes where the
library takes that path (long rows, and enough columns to fill the device)."""
import numpy as np
import pytest

import mcnla_amd as mc

pytestmark = pytest.mark.gpu


def sketch(A, order, N, l, seed=3, lda_pad=0):
    m, n = A.shape
    P = mc.Parameters().setSize(m, n).setRank(l).setOverRank(0).setNumSketch(N)
    s = mc.ColBlockGaussianProjectionSketcher(P, seed=seed)
    shape = (m + lda_pad, n) if order == "F" else (m, n + lda_pad)
    host = np.full(shape, 7.0, A.dtype, order=order)
    host[:m, :n] = A
    buf = mc.DeviceArray.from_numpy(host, order=order)
    view = mc.DeviceArray.view(buf.ptr, (m, n), A.dtype, order, ld=host.shape[0 if order == "F" else 1])
    Y = P.createCollectionQ()
    s(view, Y)
    mc.synchronize()
    return Y.numpy(), s.omega()


def check_rows(A, Y, omega, rows):
    """|Y - A Omega| is at most the rounding of the scaled operands to integers (half a unit of
    2^-58.19 of the norm, or of 2^-53 of twice the largest entry, per entry) and of the result."""
    x = A[rows].astype(np.longdouble)
    w = omega.astype(np.longdouble)
    ref = x @ w
    K = np.sqrt(np.longdouble(A.shape[1]))
    na, nw = np.sqrt((x * x).sum(1)), np.sqrt((w * w).sum(0))
    ua = np.maximum(na * 2.0 ** -58.19, np.abs(x).max(1) * 2.0 ** -53)
    uw = np.maximum(nw * 2.0 ** -58.19, np.abs(w).max(0) * 2.0 ** -53)
    bound = K * (np.outer(ua, nw) + np.outer(na, uw)) * 1.001 + np.abs(ref) * 2.0 ** -52
    err = np.abs(Y[rows] - ref)
    assert np.all(err <= bound), float((err - bound).max())


@pytest.mark.parametrize("m,n,N,l,dtype,order,pad", [
    (1000, 1000, 5, 20, np.float64, "F", 0),
    (1001, 999, 3, 33, np.float64, "F", 3),     # odd sizes and leading dimension
    (2817, 1281, 9, 31, np.float64, "C", 0),    # one row past a tile, one k past a loop body
    (1025, 1280, 1, 64, np.float64, "C", 5),
    (769, 2500, 8, 33, np.float32, "F", 1),     # 264 columns: 8 in the second tile
    (1500, 4097, 4, 16, np.float32, "C", 0),
    (12345, 2000, 10, 25, np.float64, "F", 0),  # several panels
])
def test_sketch_by_residues(m, n, N, l, dtype, order, pad):
    rng = np.random.default_rng(m + n)
    A = rng.standard_normal((m, n))
    A *= 10.0 ** rng.uniform(-6, 6, (m, 1))       # every row its own scale
    A[1] = 0.0
    A[2] *= 10.0 ** rng.uniform(-12, 0, n)        # a wide range inside a row
    A[3, 7] = 1e9 * np.abs(A[3]).max()            # one entry that dominates its row
    A[4] = np.sign(A[4])                          # every entry at the row's maximum
    A = A.astype(dtype)
    Y, omega = sketch(A, order, N, l, lda_pad=pad)
    rows = np.unique(np.r_[0:8, m // 2, 255:258, m - 3:m])
    rows = rows[rows < m]
    check_rows(A, Y, omega, rows)
    assert np.all(Y[1] == 0.0)


@pytest.mark.parametrize("scale", [1e-110, 1e100, 1e-200, 1e200])
def test_sketch_by_residues_extreme_scales(scale):
    """Norms of 1e-110 and 1e100 have a scale; 1e-200 and 1e200 leave its range and take the FP64
    product (relative accuracy of an FP64 sum)."""
    m, n, N, l = 1000, 1000, 5, 20
    rng = np.random.default_rng(5)
    A = rng.standard_normal((m, n))
    A[17] *= scale
    Y, omega = sketch(A, "F", N, l)
    rows = np.array([0, 16, 17, 18, 999])
    x, w = A[rows].astype(np.longdouble), omega.astype(np.longdouble)
    bound = np.sqrt((x * x).sum(1))[:, None] * np.sqrt((w * w).sum(0))[None, :] * (n * 2.0 ** -53)
    assert np.all(np.abs(Y[rows] - x @ w) <= bound)


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_sketch_by_residues_non_finite(value):
    m, n, N, l = 1000, 1000, 5, 20
    A = np.random.default_rng(6).standard_normal((m, n))
    A[500, 123] = value
    Y, omega = sketch(A, "F", N, l)
    with np.errstate(invalid="ignore"):
        row = A[500] @ omega
    assert np.array_equal(np.isnan(Y[500]), np.isnan(row))
    assert np.array_equal(Y[500][~np.isnan(row)], row[~np.isnan(row)])
    assert np.all(np.isfinite(np.delete(Y, 500, 0)))


def lowrank(m, n, seed, dtype, order):
    rng = np.random.default_rng(seed)
    u = rng.standard_normal((m, 60)) / np.sqrt(m) * 0.95 ** np.arange(60)
    v = rng.standard_normal((n, 60)) / np.sqrt(n)
    a = u @ v.T + 1e-3 / (np.sqrt(m) + np.sqrt(n)) * rng.standard_normal((m, n))
    return np.array(a, dtype=dtype, order=order)


@pytest.mark.parametrize("m,n,k,N,dtype,order,precision,route", [
    (10007, 1203, 20, 40, np.float64, "F", mc.PREC_F64, mc.ROUTE_SKETCH),
    (20000, 1203, 21, 33, np.float32, "C", mc.PREC_MIXED_BF16, mc.ROUTE_SKETCH),
    (30001, 1111, 20, 40, np.float32, "C", mc.PREC_F64, mc.ROUTE_GRAM_OF_A),
    (30000, 1030, 20, 40, np.float64, "F", mc.PREC_F64, mc.ROUTE_GRAM_OF_A),
])
def test_gram_by_residues(m, n, k, N, dtype, order, precision, route):
    """The solver's default plan against the same solve on the FP64 tiles (kernels bit 1): the
    Gram matrices differ in the last bits, so do sigma and the bases (condition of the kept
    directions below 1e3)."""
    A = mc.DeviceArray.from_numpy(lowrank(m, n, 2, dtype, order), order=order)
    P = mc.Parameters().setSize(m, n).setRank(k).setOverRank(10).setNumSketch(N)
    out = []
    try:
        for kernels in (0, 1):
            mc.tune_clear()
            mc.tune_set(P, dict(mc.tuning_default(), kernels=kernels), precision=precision,
                        route=route)
            s = mc.Solver(P, seed=9, precision=precision, route=route)
            s.solve(A)
            out.append((s.vectorS(), s.matrixU(), s.matrixV(), s.matrixQbar(), s.iteration()))
    finally:
        mc.tune_clear()
    a, b = out
    assert a[4] == b[4]
    # FP32 products of Qbar with A (mixed) see Qbar rounded to FP32: differences of 2^-24 where
    # the last bits of Qbar move a rounding
    tol = 1e-10 if precision == mc.PREC_F64 else 1e-6
    assert np.max(np.abs(a[0] - b[0]) / b[0]) < tol
    for i in (1, 2):
        assert np.linalg.norm(a[i] - b[i]) < 10 * tol * np.linalg.norm(b[i])
    assert np.linalg.norm(a[3] - b[3]) < 1e-9 * np.linalg.norm(b[3])


def test_residue_solve_in_a_server():
    """A solver carved from a server's arena (whose workspace may be smaller, with other panels)
    gives the bits of one that allocates its own."""
    m, n, k, N = 12000, 1500, 22, 32
    A = mc.DeviceArray.from_numpy(lowrank(m, n, 4, np.float64, "F"), order="F")
    P = mc.Parameters().setSize(m, n).setRank(k).setOverRank(10).setNumSketch(N)
    s = mc.Solver(P, seed=12)
    s.solve(A)
    need = mc.required_bytes(m, n, k, 10, N)
    results = 8 * (k + m * k + n * k + m * (k + 10)) + (1 << 20)
    with mc.Server(hbm_budget=need + results, slots=1) as srv:
        rid = srv.submit(A, m, n, k, 10, N, seed=12)
        assert srv.wait(rid, 60.0)
        r = srv.result(rid)
        assert r.ok, r.error
        np.testing.assert_array_equal(r.S.numpy(), s.vectorS())
        np.testing.assert_array_equal(r.U.numpy(), s.matrixU())
        np.testing.assert_array_equal(r.V.numpy(), s.matrixV())
        np.testing.assert_array_equal(r.Qbar.numpy(), s.matrixQbar())
