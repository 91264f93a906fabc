"""A server's workers are ready when mcnla_server_create returns: of several requests submitted at
once no worker runs all, even if each takes less time than creating a worker's streams and events
(2 to 9 ms for four workers)."""
import numpy as np
import pytest

import mcnla_amd as mc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch_max", [1, 2])
def test_first_requests_run_side_by_side(gpu, batch_max):
    m, n, k, p, N = 3000, 1000, 20, 10, 16
    rng = np.random.default_rng(3)
    a = (rng.standard_normal((m, 40)) * 0.85 ** np.arange(40)) @ rng.standard_normal((40, n))
    A = mc.DeviceArray.from_numpy(np.asfortranarray(a))
    for _ in range(4):
        with mc.Server(slots=4, hbm_budget=1 << 30, batch_max=batch_max) as srv:
            ids = [srv.submit(A, m, n, k, p, N, seed=s) for s in range(8)]
            for rid in ids:
                assert srv.wait(rid, 60.0)
            assert srv.stats()["max_running"] > 1
