"""Dense 4- to 6-qubit gates on the matrix cores (both precisions) against the
oracle: every tile width (one to eight waves, one to four column blocks per
wave), gates on the low, high and mixed tile qubits, a state smaller than a
tile, register steps between them."""
import numpy as np
import pytest

import kate_amd as K
from kate_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = {"c128": 1e-12, "c64": 2e-6}  # max-abs amplitude error, as in the other parity tests


def dense(n, count, k, seed):
    rng = np.random.default_rng(seed)
    qs = [tuple(range(k)), tuple(range(n - 1, n - 1 - k, -1))]
    qs += [tuple(int(q) for q in rng.choice(n, size=k, replace=False)) for _ in range(count)]
    return [W.Gate(W.DENSE, q, 0, W.haar_unitary(rng, 1 << k)) for q in qs]


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("n,k,tile", [(6, 5, 0), (6, 6, 0), (12, 4, 12), (12, 6, 10), (13, 5, 10), (14, 4, 10),
                                      (14, 4, 11), (14, 5, 11), (14, 6, 11), (15, 6, 12), (15, 5, 0), (15, 4, 13),
                                      (15, 5, 13), (15, 6, 13), (16, 6, 0)])
def test_dense_gates_on_matrix_cores(n, k, tile, dtype):
    gates = dense(n, 4, k, 10 * n + k) + W.random_mixed(n, 30, n, max_dense=3) + dense(n, 3, k, n)
    with K.Simulator(K.Circuit(n, gates), dtype=dtype, tile_qubits=tile) as sim:
        sim.execute()
        assert np.max(np.abs(sim.state() - O.simulate(n, gates))) <= TOL[dtype]
