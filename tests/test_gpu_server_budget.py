"""A request that fits the server's memory without matrix-core operands (twice
the size of the gate as given) is served, on the VALU."""
import numpy as np
import pytest

import kate_amd as K
from kate_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["c128", "c64"])
def test_request_near_the_budget(gpu, dtype):
    n, count = 12, 150
    rng = np.random.default_rng(1)
    gates = [W.Gate(W.DENSE, tuple(int(q) for q in rng.choice(n, size=6, replace=False)), 0, W.haar_unitary(rng, 64))
             for _ in range(count)]
    # the gates as given, and 2 MiB for the state, the sums' scratch and the plan
    budget = count * 64 * 64 * (16 if dtype == "c128" else 8) + (2 << 20)
    c, masks = K.Circuit(n, gates), [1, 6, 2049]
    with K.Simulator(c, dtype=dtype) as sim, K.Server(dtype=dtype, hbm_budget_bytes=budget) as srv:
        sim.execute()
        z, _ = srv.wait(srv.submit(c, masks))
        # 150 gates of 128 rounded products an amplitude, errors of either sign:
        # 2 sqrt(150 * 128) units of rounding in each of the two forms
        unit = 2.0 ** (-53 if dtype == "c128" else -24)
        assert np.max(np.abs(z - sim.expect_z(masks))) <= 4 * (150 * 128) ** 0.5 * unit
