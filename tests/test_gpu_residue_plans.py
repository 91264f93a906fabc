"""An FP64 product by residues gives the same bits however its rows and K are cut (gemm_residue.hip):
workspaces of different sizes take other panels and other K ranges.  The operands are orthogonal to
2^-20 of their norms, so that the sums are small beside the moduli's product: there the FP64
arithmetic of the reconstruction would show which residues it was given."""
import contextlib
import ctypes

import numpy as np
import pytest

import mcnla_amd as mc
from mcnla_amd import _lib
import residue

pytestmark = pytest.mark.gpu


def plans(a):
    """Workspace sizes from the largest that is of use down, each of another plan."""
    limit, out = 2 << 30, []
    while len(out) < 8:
        size = residue.workspace(a, limit)
        if size == 0:
            break
        out.append(size)
        limit = min(size - 1, int(0.85 * size))
    return out


@pytest.mark.parametrize("m,n,k,dtype,order", [
    (700, 300, 6000, np.float64, "F"),
    (700, 300, 6000, np.float32, "C"),
    (1500, 333, 9001, np.float64, "C"),
])
def test_product_of_any_plan(m, n, k, dtype, order):
    rng = np.random.default_rng(m + k)
    A = rng.standard_normal((m, k)).astype(dtype)
    q = np.linalg.qr(A.astype(np.float64).T)[0]
    B = rng.standard_normal((k, n))
    B = B - q @ (q.T @ B) + 2.0 ** -20 * rng.standard_normal((k, n))
    dA = mc.DeviceArray.from_numpy(A, order=order)
    dB = mc.DeviceArray.from_numpy(B, order="C")
    sizes = plans(residue.args(dA, dB))
    assert len(sizes) >= 3
    results = [residue.product(dA, dB, size) for size in sizes]
    assert all(flag == 0 for _, flag in results)
    for c, _ in results[1:]:
        np.testing.assert_array_equal(c, results[0][0])


@pytest.mark.parametrize("m,k,dtype,order", [
    (300, 60000, np.float64, "F"), (600, 20001, np.float32, "F"), (260, 9000, np.float64, "C"),
])
def test_symmetric_product_of_any_plan(m, k, dtype, order):
    rng = np.random.default_rng(m + k)
    q = np.linalg.qr(rng.standard_normal((k, m)))[0].T
    A = (q + 2.0 ** -20 / np.sqrt(k) * rng.standard_normal((m, k))).astype(dtype)
    dA = mc.DeviceArray.from_numpy(A, order=order)
    sizes = plans(residue.args(dA))
    assert len(sizes) >= 3
    results = [residue.product(dA, limit=size) for size in sizes]
    assert all(flag == 0 for _, flag in results)
    for c, _ in results[1:]:
        np.testing.assert_array_equal(c, results[0][0])
    np.testing.assert_array_equal(results[0][0], results[0][0].T)


@pytest.mark.parametrize("precision,route", [
    (mc.PREC_F64, mc.ROUTE_SKETCH), (mc.PREC_MIXED_BF16, mc.ROUTE_SKETCH),
    (mc.PREC_F64, mc.ROUTE_GRAM_OF_A),
])
def test_solver_holds_what_it_reports(precision, route):
    """A solver's products by residues work in memory it has anyway: it holds what required_bytes
    says, and on the FP64 sketch route at most the partials that a sketch on the FP64 tiles would
    take for its last rows."""
    m, n, k, p, N = 60000, 3000, 20, 12, 48
    P = mc.Parameters().setSize(m, n).setRank(k).setOverRank(p).setNumSketch(N)
    s = mc.Solver(P, precision=precision, route=route)
    tail = 0
    if precision == mc.PREC_F64 and route == mc.ROUTE_SKETCH:
        splits = ctypes.c_int64()
        main = residue.function("gemm_f64_dma_tail", ctypes.c_int64, *[ctypes.c_int64] * 3,
                                ctypes.c_void_p)(m, (k + p) * N, n, ctypes.byref(splits))
        tail = 8 * (m - main) * (k + p) * N * splits.value
    required = mc.required_bytes(m, n, k, p, N, precision=precision, route=route)
    assert s.workspace_bytes() <= required + tail


def decaying(m, n):
    rng = np.random.default_rng(8)
    a = (rng.standard_normal((m, 60)) * 0.95 ** np.arange(60)) @ rng.standard_normal((60, n))
    return a + 1e-3 * rng.standard_normal((m, n))


@pytest.mark.parametrize("m,n,k,p,N", [(6000, 9000, 20, 12, 50), (30000, 2500, 50, 10, 32)])
def test_solve_in_a_server(m, n, k, p, N):
    """An FP64 solve whose Gram (and sketch, in the first case) run by residues gives the same bits
    in a server's region and in a solver's own memory, whatever workspace either has."""
    A = mc.DeviceArray.from_numpy(decaying(m, n), order="F")
    P = mc.Parameters().setSize(m, n).setRank(k).setOverRank(p).setNumSketch(N)
    s = mc.Solver(P, seed=12)
    s.solve(A)
    assert residue.solver_paths(s)[1]
    need = mc.required_bytes(m, n, k, p, N)
    results = 8 * (k + m * k + n * k + m * (k + p)) + (1 << 20)
    with mc.Server(hbm_budget=need + results, slots=1) as srv:
        rid = srv.submit(A, m, n, k, p, N, seed=12)
        assert srv.wait(rid, 60.0)
        r = srv.result(rid)
        assert r.ok, r.error
        for x, y in ((r.S, s.vectorS()), (r.U, s.matrixU()), (r.V, s.matrixV()),
                     (r.Qbar, s.matrixQbar())):
            np.testing.assert_array_equal(x.numpy(), y)


@pytest.fixture
def untuned():
    mc.tune_clear()
    yield
    mc.tune_clear()


@pytest.mark.parametrize("m,n,k,p,N,sketch", [
    (6000, 9000, 20, 12, 50, True),    # with 576 the partials could not hold the packed Omega
    (40000, 1000, 50, 10, 32, False),  # with 9216 the Gram takes other panels and ranges
])
def test_tuned_plan_keeps_the_route(untuned, m, n, k, p, N, sketch):
    """The Gram's split target changes neither the route of an FP64 sketch and its Gram nor a bit
    of the results."""
    A = mc.DeviceArray.from_numpy(decaying(m, n), order="F")
    P = mc.Parameters().setSize(m, n).setRank(k).setOverRank(p).setNumSketch(N)
    out = []
    for gram in (2304, 576, 9216):
        mc.tune_set(P, dict(mc.tuning_default(), gram=gram), route=mc.ROUTE_SKETCH)
        s = mc.Solver(P, seed=9, route=mc.ROUTE_SKETCH)
        s.solve(A)
        assert residue.solver_paths(s) == (sketch, True)
        out.append((s.vectorS(), s.matrixU(), s.matrixV(), s.matrixQbar()))
    for other in out[1:]:
        for x, y in zip(out[0], other):
            np.testing.assert_array_equal(x, y)


@contextlib.contextmanager
def little_memory(left):
    """All but about `left` bytes of the device's memory taken."""
    held = []
    try:
        while (free := mc.mem_info()[0]) > left + (64 << 20):
            held.append(mc.DeviceArray((min(free - left, 16 << 30) // 8,)))
        yield
    finally:
        for x in held:
            x.free()


def test_sketcher_with_little_memory():
    """A sketcher stage takes at most an eighth of the free memory for its residue workspace, and
    gives the same bits in a smaller one."""
    m, n, l, N = 4001, 4099, 41, 25
    A = mc.DeviceArray.from_numpy(np.random.default_rng(4).standard_normal((m, n)), order="F")
    P = mc.Parameters().setSize(m, n).setRank(l).setOverRank(0).setNumSketch(N)

    def sketch():
        s = mc.ColBlockGaussianProjectionSketcher(P, seed=3).initialize()
        before = mc.mem_info()[0]
        s(A, Q)
        mc.synchronize()
        assert residue.sketcher_path(s)
        return Q.numpy(), before, before - mc.mem_info()[0]
    Q = P.createCollectionQ()
    y, _, taken = sketch()
    assert taken > 400 << 20
    with little_memory(5 << 29):
        z, before, taken = sketch()
    assert taken <= before // 8 + (4 << 20)
    np.testing.assert_array_equal(y, z)


def test_autotune_without_memory(untuned):
    """Candidate plans that there is no memory for: the tuner reports it, and the solver goes on
    with the plan it had."""
    m, n, k, p, N = 30000, 2500, 50, 10, 32
    A = mc.DeviceArray.from_numpy(decaying(m, n), order="F")
    P = mc.Parameters().setSize(m, n).setRank(k).setOverRank(p).setNumSketch(N)
    s = mc.Solver(P, seed=12)
    s.solve(A)
    before, plan = (s.vectorS(), s.matrixU(), s.matrixV(), s.matrixQbar()), s.tuning()
    with little_memory(1 << 29):
        with pytest.raises(mc.McnlaError) as e:
            s.autotune(A, reps=1)
        assert e.value.status == _lib.ERR_NOMEM
        assert s.tuning() == plan
        s.solve(A)
        for x, y in zip(before, (s.vectorS(), s.matrixU(), s.matrixV(), s.matrixQbar())):
            np.testing.assert_array_equal(x, y)
