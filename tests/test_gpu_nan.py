"""A NaN in a gate reaches the amplitudes, in streamed programs too (a 1-qubit
gate in a program with CRk)."""
import numpy as np
import pytest

import kate_amd as K
from kate_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("entry", range(4))
def test_nan_entry_reaches_the_state(gpu, entry, dtype):
    n = 8
    u = W.haar_unitary(np.random.default_rng(entry), 2)
    u.reshape(-1)[entry] = np.nan
    # from |0...0> every Hadamard layer spreads what the gate left in one half
    # of the state to all of it
    layer = [W.Gate(W.H, (q,)) for q in range(n)]
    gates = layer + [W.Gate(W.CRK, (0, 1), 3), W.Gate(W.DENSE, (2,), 0, u)] + layer
    with K.Simulator(K.Circuit(n, gates), dtype=dtype) as sim:
        sim.execute()
        assert np.isnan(sim.state()).all()
