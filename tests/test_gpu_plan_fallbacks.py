"""The branches of the planner and the kernels that ordinary circuits do not
reach: what a streamed program falls back to, wide dense gates kept off the
matrix cores, sums gathered over several chunks a workgroup, and states on both
sides of the plan-ahead line held to the rounding of their gates."""
import numpy as np
import pytest

import kate_amd as K
from kate_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu

UNIT = {"c128": 2.0 ** -53, "c64": 2.0 ** -24}


def check(n, gates, dtype, tp=None, **kw):
    """Norm of the error against the oracle.  A gate of k qubits rounds an
    amplitude through 2^k products, in our order and in the oracle's: errors of
    either sign, 2 * sqrt(2^k) units of the state's norm a gate in each, added
    as independent ones over the gates."""
    want = O.simulate(n, gates, tp)
    tol = 4 * np.sqrt(sum(2.0 ** len(g.qubits) for g in gates)) * UNIT[dtype]
    with K.Simulator(K.Circuit(n, gates), dtype=dtype, **kw) as sim:
        for _ in range(2):
            sim.execute(tp)
            assert np.linalg.norm(sim.state() - want) <= tol * np.linalg.norm(want)
        return sim.describe()


def phases(n, count, seed):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(count):
        pair = tuple(int(q) for q in rng.choice(n, 2, replace=False))
        kind = int(rng.integers(0, 3))
        out.append(W.Gate(W.H, pair[:1]) if kind == 0 else
                   W.Gate(W.DENSE, pair[:1], 0, W.rx(float(rng.uniform(0, 3)))) if kind == 1 else
                   W.Gate(W.CRK, pair, int(rng.integers(1, 12))))
    return out


def dense(n, count, k, seed):
    rng = np.random.default_rng(seed)
    return [W.Gate(W.DENSE, tuple(int(q) for q in rng.choice(n, size=k, replace=False)), 0, W.haar_unitary(rng, 1 << k))
            for _ in range(count)]


@pytest.mark.parametrize("dtype", ["c128", "c64"])
def test_more_phases_than_a_pass_holds(gpu, dtype):
    assert " stream" in check(12, phases(12, 600, 1), dtype)
    # the fallback is the plan without streams, as an explicit tile size gives it
    c = K.Circuit(12, phases(12, 1600, 1))
    states = []
    for kw in ({}, {"tile_qubits": 12}):
        with K.Simulator(c, dtype=dtype, **kw) as sim:
            sim.execute()
            assert " stream" not in sim.describe()
            states.append(sim.state())
    assert np.array_equal(*states)
    assert np.max(np.abs(states[0] - O.simulate(12, phases(12, 1600, 1)))) <= {"c128": 1e-12, "c64": 2e-6}[dtype]


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("n", [6, 12, 15])
def test_gate_that_is_not_unitary_among_phases(gpu, n, dtype):
    m = np.array([[0.9, 0.3j], [0.2, 1.1]], dtype=np.complex128)
    gates = W.layered(n, 1, n) + W.qft(n)
    assert " stream" in check(n, gates, dtype)
    gates.insert(len(gates) // 2, W.Gate(W.DENSE, (n // 2,), 0, m))
    assert " stream" not in check(n, gates, dtype)


@pytest.mark.parametrize("dtype,mb", [("c128", 4), ("c128", 3), ("c64", 4)])
@pytest.mark.parametrize("tile", [10, 11, 12, 13])
def test_wide_gates_on_the_valu(gpu, tile, dtype, mb, monkeypatch):
    monkeypatch.setenv("KATE_DESCRIBE_OPS", "1")
    n = 15
    gates = (dense(n, 8, 5, tile) + W.random_mixed(n, 30, tile, max_dense=4) + dense(n, 4, 6, tile) +
             dense(n, 3, 7, tile) + dense(n, 4, 5, tile + 1))
    text = check(n, gates, dtype, tile_qubits=tile, micro_bits=mb, matrix5=False)
    assert text.count(" generic ") >= 19 and " mfma" not in text


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("n,k", [(8, 8), (10, 9), (10, 10), (11, 11), (14, 7)])
def test_gates_wider_than_the_matrix_cores_take(gpu, n, k, dtype):
    check(n, W.layered(n, 1, k) + dense(n, 2, k, n) + dense(n, 3, min(6, k), n), dtype)


@pytest.mark.parametrize("tile,mb", [(10, 4), (11, 4), (12, 4), (13, 4), (10, 3), (12, 3)])
def test_batches_of_wide_gates(gpu, tile, mb):
    sizes = [10, 12, 13, 14]
    circuits = [(n, W.layered(n, 1, n) + dense(n, 4, 5, n) + dense(n, 2, 6, n) + W.layered(n, 1, n + 1)) for n in sizes]
    with K.Batch([K.Circuit(n, g) for n, g in circuits], dtype="c128", tile_qubits=tile, micro_bits=mb) as b:
        b.run()
        z, norms = b.expect_z()
    for (n, g), zc, norm in zip(circuits, z, norms):
        want = O.expect_z(n, O.simulate(n, g), [1 << q for q in range(n)])
        tol = 8 * np.sqrt(sum(2.0 ** len(x.qubits) for x in g)) * UNIT["c128"]  # twice the state's
        assert np.max(np.abs(zc - want)) <= tol and abs(norm - 1) <= tol


@pytest.mark.parametrize("n,dtype", [(22, "c128"), (24, "c64"), (25, "c64")])
def test_sums_through_pending_permutations(gpu, n, dtype):
    """Up to 2^11 chunks of 4096 amplitudes a workgroup reads one, at 24 qubits
    two, at 25 four: gathered through the trailing CNOTs and read in place."""
    with K.Simulator(K.Circuit(n, W.layered(n, 3, n)), dtype=dtype, scatter=False, defer=True) as sim:
        assert " micro=0 " in sim.describe().splitlines()[-1]
        gathered = sim.execute()
        sim.state()  # runs the trailing passes
        assert np.max(np.abs(gathered - sim.measure_proba())) < 1e-9


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("n", [10, 13, 20, 21, 22])
@pytest.mark.parametrize("kind", ["layered", "qft", "brickwork"])
def test_both_sides_of_the_plan_ahead_line(gpu, kind, n, dtype):
    gates = {"layered": lambda: W.layered(n, 2, 3), "qft": lambda: W.qft(n), "brickwork": lambda: W.brickwork(n, 4, 7)}
    check(n, gates[kind](), dtype, W.basis_input(n, 5) if kind == "qft" else None)
