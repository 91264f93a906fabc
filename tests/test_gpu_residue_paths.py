"""FP64 products by residues (gemm_residue.hip) at the edges of their tiles, panels and loops, each
run asserted to have taken that path: the product by itself, the sketcher stage, and solves whose
operands have rows without a scale (the flag and the gated FP64 product behind it)."""
import numpy as np
import pytest

import mcnla_amd as mc
import residue

pytestmark = pytest.mark.gpu


def device(a, order, pad=0):
    """The matrix on the device, with a leading dimension `pad` past its own."""
    m, n = a.shape
    host = np.full((m + pad, n) if order == "F" else (m, n + pad), 7.0, a.dtype, order=order)
    host[:m, :n] = a
    buf = mc.DeviceArray.from_numpy(host, order=order)
    view = mc.DeviceArray.view(buf.ptr, (m, n), a.dtype, order, ld=host.shape[0 if order == "F" else 1])
    view.buf = buf
    return view


def rows_of(m, n, dtype):
    """Rows of every kind: their own scales, a zero one, a wide range inside, one entry that
    dominates, every entry at the maximum."""
    rng = np.random.default_rng(m + n)
    A = rng.standard_normal((m, n))
    A *= 10.0 ** rng.uniform(-6, 6, (m, 1))
    A[1] = 0.0
    A[2] *= 10.0 ** rng.uniform(-12, 0, n)
    A[3, 7] = 1e9 * np.abs(A[3]).max()
    A[4] = np.sign(A[4])
    return A.astype(dtype)


def check(A, B, C, rows):
    """|C - A B| in some rows is at most what the rounding of the scaled operands to integers gives
    (half a unit of 2^-58.19 of the norm, or of 2^-53 of twice the largest entry, per entry), the
    reconstruction's 2^-70 of the norms and the rounding of the result."""
    x, w = A[rows].astype(np.longdouble), B.astype(np.longdouble)
    ref = x @ w
    na, nw = np.sqrt((x * x).sum(1)), np.sqrt((w * w).sum(0))
    ua = np.maximum(na * 2.0 ** -58.19, np.abs(x).max(1) * 2.0 ** -53)
    uw = np.maximum(nw * 2.0 ** -58.19, np.abs(w).max(0) * 2.0 ** -53)
    bound = (np.outer(ua, np.abs(w).sum(0)) + np.outer(np.abs(x).sum(1), uw)) * 1.001 + \
        np.outer(na, nw) * 2.0 ** -68 + np.abs(ref) * 2.0 ** -53
    err = np.abs(C[rows] - ref)
    assert np.all(err <= bound), float((err - bound).max())


def some_rows(m):
    rows = np.unique(np.r_[0:8, m // 2, 127:130, 255:258, m - 3:m])
    return rows[(rows >= 0) & (rows < m)]


@pytest.mark.parametrize("m,n,k,dtype,order,pad", [
    (256, 256, 640, np.float64, "F", 0),     # one tile, one loop body
    (257, 255, 641, np.float64, "F", 1),     # one row past a tile, one k past a loop body
    (257, 257, 639, np.float64, "C", 1),
    (5, 1, 64, np.float64, "C", 0),          # far less than a tile
    (6, 3, 1, np.float64, "F", 0),
    (300, 600, 1000, np.float32, "F", 3),
    (511, 100, 2000, np.float32, "C", 5),
    (3000, 520, 5001, np.float64, "F", 0),   # several K ranges
])
def test_product(m, n, k, dtype, order, pad):
    if m >= 8 and k >= 8:
        A = rows_of(m, k, dtype)
    else:
        A = np.random.default_rng(k).standard_normal((m, k)).astype(dtype)
    B = np.random.default_rng(n).standard_normal((k, n))
    B[:, 0] = 0.0
    C, flag = residue.product(device(A, order, pad), device(B, "C", pad))
    assert flag == 0
    check(A, B, C, some_rows(m))
    assert np.all(C[:, 0] == 0.0)


@pytest.mark.parametrize("m,k,dtype,order,pad", [
    (256, 640, np.float64, "F", 0), (257, 641, np.float64, "F", 1), (65, 3000, np.float64, "C", 3),
    (513, 2001, np.float32, "F", 1), (300, 999, np.float32, "C", 0), (1, 70, np.float64, "F", 0),
])
def test_symmetric_product(m, k, dtype, order, pad):
    A = rows_of(m, k, dtype) if m >= 8 else np.ones((m, k), dtype)
    C, flag = residue.product(device(A, order, pad))
    assert flag == 0
    check(A, A.T.astype(np.float64), C, np.arange(m))
    np.testing.assert_array_equal(C, C.T)


@pytest.mark.parametrize("value,scaled", [(1e-110, True), (1e100, True), (1e-200, False),
                                          (1e200, False), (np.nan, False), (np.inf, False),
                                          (-np.inf, False)])
@pytest.mark.parametrize("order", ["F", "C"])
def test_flag(value, scaled, order):
    """A row whose norm leaves [2^-400, 2^400], or with a non-finite entry, raises the flag, in
    either operand and at either end; norms inside do not."""
    m, n, k = 300, 270, 700
    rng = np.random.default_rng(2)
    A, B = rng.standard_normal((m, k)), rng.standard_normal((k, n))
    for which, at in ((0, 0), (0, m - 1), (1, 0), (1, n - 1)):
        a, b = A.copy(), B.copy()
        line = a[at] if which == 0 else b[:, at]
        if np.isfinite(value):
            line *= value
        else:
            line[k - 1] = value
        c, flag = residue.product(device(a, order), device(b, "C"))
        assert (flag == 0) == scaled, (which, at)
        assert np.all(np.isnan(c)) != scaled  # nothing is written behind a raised flag
        if which == 0:
            c, flag = residue.product(device(a, order))
            assert (flag == 0) == scaled, at
            assert np.all(np.isnan(c)) != scaled


def sketch(A, order, N, l, pad=0):
    m, n = A.shape
    P = mc.Parameters().setSize(m, n).setRank(l).setOverRank(0).setNumSketch(N)
    s = mc.ColBlockGaussianProjectionSketcher(P, seed=3).initialize()
    Y = P.createCollectionQ()
    view = device(A, order, pad)
    s(view, Y)
    mc.synchronize()
    assert residue.sketcher_path(s)
    return Y.numpy(), s.omega()


@pytest.mark.parametrize("m,n,N,l,dtype,order,pad", [
    (4001, 4099, 41, 25, np.float64, "F", 0),
    (4001, 4099, 41, 25, np.float64, "C", 1),
    (4001, 4099, 25, 41, np.float32, "F", 3),
    (4099, 4001, 41, 25, np.float32, "C", 5),
    (12289, 3001, 103, 10, np.float64, "F", 0),  # several panels of A
])
def test_sketch(m, n, N, l, dtype, order, pad):
    A = rows_of(m, n, dtype)
    Y, omega = sketch(A, order, N, l, pad)
    check(A, omega, Y, some_rows(m))
    assert np.all(Y[1] == 0.0)


@pytest.mark.parametrize("scale", [1e-110, 1e100, 1e-200, 1e200])
def test_sketch_with_an_extreme_row(scale):
    """1e-110 and 1e100 have a scale; 1e-200 and 1e200 take the FP64 product (whose sums round to
    n eps of the products' magnitudes)."""
    m, n = 4001, 4099
    A = np.random.default_rng(5).standard_normal((m, n))
    A[17] *= scale
    Y, omega = sketch(A, "F", 41, 25)
    rows = np.array([0, 16, 17, 18, m - 1])
    x, w = A[rows].astype(np.longdouble), omega.astype(np.longdouble)
    assert np.all(np.abs(Y[rows] - x @ w) <= n * 2.0 ** -53 * (np.abs(x) @ np.abs(w)))


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_sketch_with_a_non_finite_entry(value):
    m, n = 4001, 4099
    A = np.random.default_rng(6).standard_normal((m, n))
    A[500, 123] = value
    Y, omega = sketch(A, "F", 41, 25)
    with np.errstate(invalid="ignore"):
        row = A[500] @ omega
    assert np.array_equal(np.isnan(Y[500]), np.isnan(row))
    assert np.array_equal(Y[500][~np.isnan(row)], row[~np.isnan(row)])
    rows = np.array([0, 499, 501, m - 1])
    x, w = A[rows].astype(np.longdouble), omega.astype(np.longdouble)
    assert np.all(np.abs(Y[rows] - x @ w) <= n * 2.0 ** -53 * (np.abs(x) @ np.abs(w)))


def lowrank(m, n, dtype, order):
    rng = np.random.default_rng(m + n)
    u = rng.standard_normal((m, 60)) / np.sqrt(m) * 0.95 ** np.arange(60)
    a = u @ (rng.standard_normal((n, 60)) / np.sqrt(n)).T
    a += 1e-3 / (np.sqrt(m) + np.sqrt(n)) * rng.standard_normal((m, n))
    return np.array(a, dtype=dtype, order=order)


@pytest.mark.parametrize("order", ["F", "C"])
@pytest.mark.parametrize("scale", [1e-200, 1e200, np.nan])
def test_gram_of_a_with_a_column_without_a_scale(scale, order):
    """A'A by residues, one column of A too small or too large for a scale (then the FP64 product
    replaces it: sigma as on the FP64 tiles, to the rounding of the sums) or not finite (an error on
    either)."""
    m, n, k, N = 30000, 1030, 20, 40
    a = lowrank(m, n, np.float64, order)
    if np.isnan(scale):
        a[m - 1, 5] = scale
    elif scale < 1:
        a[:, 5] *= scale
    else:
        a *= scale  # every column
    A = mc.DeviceArray.from_numpy(a, order=order)
    P = mc.Parameters().setSize(m, n).setRank(k).setOverRank(10).setNumSketch(N)
    out = []
    try:
        for kernels in (0, 1):
            mc.tune_clear()
            mc.tune_set(P, dict(mc.tuning_default(), kernels=kernels), route=mc.ROUTE_GRAM_OF_A)
            s = mc.Solver(P, seed=9, route=mc.ROUTE_GRAM_OF_A)
            try:
                s.solve(A)
                status = 0
            except mc.McnlaError as e:
                status = e.status
            assert residue.solver_paths(s)[1] == (kernels == 0)
            out.append((status, s.vectorS() if status == 0 else None))
    finally:
        mc.tune_clear()
    assert out[0][0] == out[1][0]
    if scale < 1:
        assert out[0][0] == 0
        assert np.max(np.abs(out[0][1] - out[1][1]) / out[1][1]) < 1e-10
    else:
        assert out[0][0] != 0


@pytest.mark.parametrize("kind", ["lognormal", "cauchy", "outliers"])
def test_gram_of_a_with_spread_columns(kind):
    """Columns whose entries spread over many orders of magnitude: the residue product holds the
    small ones to fewer bits than FP64 does, and bounds the error of an entry of A'A by the two
    columns' norms alone.  Sigma takes no harm: either product's error is below m 2^-53 of the
    columns' norms, so sigma_j differs by at most m 2^-53 (||A||_F / sigma_j)^2 of itself."""
    m, n, k, N = 40000, 1200, 20, 40
    rng = np.random.default_rng(7)
    if kind == "lognormal":
        a = np.exp(3 * rng.standard_normal((m, n))) * rng.choice([-1.0, 1.0], (m, n))
    elif kind == "cauchy":
        a = rng.standard_normal((m, n)) / rng.standard_normal((m, n))
    else:
        a = rng.standard_normal((m, n))
        a[rng.permutation(m)[:n], np.arange(n)] = 1e8 * 0.9 ** np.arange(n) + 1e3
    A = mc.DeviceArray.from_numpy(a, order="C")
    P = mc.Parameters().setSize(m, n).setRank(k).setOverRank(10).setNumSketch(N)
    out = []
    try:
        for kernels in (0, 1):
            mc.tune_clear()
            mc.tune_set(P, dict(mc.tuning_default(), kernels=kernels), route=mc.ROUTE_GRAM_OF_A)
            s = mc.Solver(P, seed=9, route=mc.ROUTE_GRAM_OF_A)
            s.solve(A)
            assert residue.solver_paths(s)[1] == (kernels == 0)
            out.append(s.vectorS())
    finally:
        mc.tune_clear()
    bound = m * 2.0 ** -53 * (np.linalg.norm(a) / out[1]) ** 2
    assert np.all(np.abs(out[0] - out[1]) <= bound * out[1])
