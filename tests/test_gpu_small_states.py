"""States of fewer than 12 qubits run in a tile of their own size (10 or 11
qubits, one to two waves) inside a buffer of 4096 amplitudes: every gate kind
and both inputs against the oracle, amplitudes, norm and Z strings, streamed
passes included."""
import numpy as np
import pytest

import kate_amd as K
from kate_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu

KINDS = {"layered": lambda n: W.layered(n, 6, 3), "qft": W.qft, "mixed": lambda n: W.random_mixed(n, 60, 5, min(3, n)),
         "brickwork": lambda n: W.brickwork(n, 6, 7)}


@pytest.mark.parametrize("dtype,tol", [("c128", 1e-12), ("c64", 2e-5)])
@pytest.mark.parametrize("n", [1, 4, 5, 9, 10, 11, 12])
@pytest.mark.parametrize("kind", sorted(KINDS))
def test_small_states(gpu, kind, n, dtype, tol):
    print("small", kind, n, dtype, flush=True)
    if n < 3 and kind != "layered":
        pytest.skip("needs three qubits")
    gates = KINDS[kind](n)
    masks = [0, 1, (1 << n) - 1]
    for tp in (None, W.basis_input(n, (1 << n) - 1)):
        want = O.simulate(n, gates, tp)
        with K.Simulator(K.Circuit(n, gates), dtype=dtype) as sim:
            for _ in range(2):
                sim.execute(tp)
                assert np.max(np.abs(sim.state() - want)) < tol
                assert np.max(np.abs(sim.expect_z(masks) - O.expect_z(n, want, masks))) < tol
