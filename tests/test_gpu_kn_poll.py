"""The KN loop that reads its convergence flags one chunk (8 iterations) behind its launches, at the
ends of chunks: iteration limits on both sides of them, never converging or converging within the
last chunk, against the loop that waits for every chunk (the one recorded as graphs), bit for bit."""
import numpy as np
import pytest

import mcnla_amd as mc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("limit", [1, 7, 8, 9, 16, 17, 256])
@pytest.mark.parametrize("tol", [0.0, 1e-1, 1e-4])
def test_iteration_limits(limit, tol):
    if limit == 256 and tol == 0.0:
        limit = 40
    rng = np.random.default_rng(limit)
    A = mc.DeviceArray.from_numpy(np.asfortranarray(
        rng.standard_normal((300, 120)) * 0.9 ** np.arange(120)))
    P = mc.Parameters().setSize(300, 120).setRank(6).setOverRank(4).setNumSketch(7)
    out = []
    for graph in (False, True):
        s = mc.Solver(P, seed=3, max_iteration=limit, tolerance=tol, graph=graph)
        for _ in range(2):  # the second solve replays; both sets of flags hold old values
            s.solve(A)
            out.append((s.iteration(), s.vectorS(), s.matrixU(), s.matrixQbar()))
    for got in out[1:]:
        assert got[0] == out[0][0]
        for x, y in zip(got[1:], out[0][1:]):
            assert np.array_equal(x, y)
    if tol == 0.0:
        assert out[0][0] == limit
