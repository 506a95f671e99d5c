"""Streamed passes (1-qubit, CNOT and CRk gates on k_stream) against the
oracle, at the sizes where they change: a padded state, one tile, one more
qubit, several passes (phases of tile and rest qubits, relabelled, in place,
through the trailing permutation) and programs with swaps."""
import numpy as np
import pytest

import kate_amd as K
from kate_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# max-abs amplitude error, as in the other parity tests
TOL = {"c128": 1e-12, "c64": 2e-6}


def circuit(n, ngates, seed):
    """Haar 1-qubit gates, H, X (a rotation by pi, no rotation at all), CNOT,
    and CRk up to phases below the rounding of either type."""
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(ngates):
        kind = int(rng.integers(0, 7))
        pair = tuple(int(q) for q in rng.choice(n, 2, replace=False))
        if kind == 0:
            out.append(W.Gate(W.DENSE, pair[:1], 0, W.haar_unitary(rng, 2)))
        elif kind == 1:
            out.append(W.Gate(W.H, pair[:1]))
        elif kind == 2:
            out.append(W.Gate(W.DENSE, pair[:1], 0, np.array([[0, 1], [1, 0]], dtype=np.complex128)))
        elif kind == 3:
            out.append(W.Gate(W.CNOT, pair))
        else:
            out.append(W.Gate(W.CRK, pair, int(rng.integers(1, 40))))
    return out


def angles(n, seed):
    rng = np.random.default_rng(seed)
    return np.column_stack([rng.uniform(0.05, 0.95, n), rng.uniform(0, 6.2, n)])


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("n,product,kw", [(3, True, {}), (12, False, {}), (13, True, {}), (16, False, {}),
                                          (16, True, {"relabel": False}), (17, True, {"scatter": False}),
                                          (18, True, {}), (18, False, {"reorder": False})])
def test_streamed_circuits(n, product, kw, dtype):
    for seed, gates in ((1, circuit(n, 160, n)), (2, W.layered(n, 1, n) + W.qft(n))):
        tp = angles(n, seed) if product else None
        ref = O.simulate(n, gates, tp)
        with K.Simulator(K.Circuit(n, gates), dtype=dtype, **kw) as sim:
            assert " stream" in sim.describe()
            pr = sim.execute(tp)
            err = np.max(np.abs(sim.state() - ref))
            if dtype == "c128":
                assert np.max(np.abs(pr - O.measure(n, ref))) < 1e-9
        assert err <= TOL[dtype]


@pytest.mark.parametrize("dtype", ["c128", "c64"])
def test_streamed_swap_program(dtype):
    n = 17
    gates = circuit(n, 200, 5)
    with K.Simulator(K.Circuit(n, gates).schedule().group(8).allocate(2), dtype=dtype) as sim:
        assert " stream" in sim.describe() and sim.timings()["remap_passes"] > 0
        sim.execute()
        assert np.max(np.abs(sim.state() - O.simulate(n, gates))) <= TOL[dtype]


def test_served_streamed_requests():
    """In place below 22 qubits, relabelled on two buffers from there on."""
    with K.Server(dtype="c128", hbm_budget_bytes=1 << 30) as srv:
        work = []
        for n in (12, 15, 22):
            gates, tp = W.qft(n), angles(n, n)
            masks = [int(m) for m in W.zstring_masks(n, 6, n)]
            work.append((n, gates, tp, masks, srv.submit(K.Circuit(n, gates), masks, tp)))
        for n, gates, tp, masks, rid in work:
            z, _ = srv.wait(rid)
            with K.Simulator(K.Circuit(n, gates), tile_qubits=12) as sim:  # unstreamed
                sim.execute(tp)
                assert np.max(np.abs(z - sim.expect_z(masks))) <= 1e-12
