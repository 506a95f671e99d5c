"""The planner streams a program with CRk gates only where that is the cheaper
form: QFTs and rings of CRk, not layers with a few CRk among them."""
import numpy as np
import pytest

import kate_amd as K
from kate_amd import workloads as W


def with_crk(gates, n, count):
    rng = np.random.default_rng(count)
    for _ in range(count):
        pair = tuple(int(q) for q in rng.choice(n, 2, replace=False))
        gates.insert(int(rng.integers(0, len(gates) + 1)), W.Gate(W.CRK, pair, int(rng.integers(1, 10))))
    return gates


def ladders(n, layers):
    one = [W.Gate(W.H, (q,)) for q in range(n)] + [W.Gate(W.CNOT, (q + 1, q)) for q in range(n - 1)]
    return one * layers


def rings(n, layers):
    out = []
    for i in range(layers):
        out += [W.Gate(W.CRK, (q, (q + 1) % n), 3) for q in range(n)]
        out += [g for g in W.layered(n, 1, i) if g.id == W.DENSE]
    return out


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("n", [22, 25, 28])
@pytest.mark.parametrize("kind,count", [("layered", 1), ("layered", 16), ("ladders", 1), ("ladders", 16)])
def test_few_phases_among_layers(kind, count, n, dtype):
    gates = W.layered(n, 10, 3) if kind == "layered" else ladders(n, 10)
    _, _, plain = K.Circuit(n, gates).plan(dtype)
    _, _, text = K.Circuit(n, with_crk(gates, n, count)).plan(dtype)
    assert " light" in plain and " stream" not in text and " light" in text


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("n", [4, 12, 16, 25, 28])
def test_many_phases(n, dtype):
    for gates in (W.qft(n), W.layered(n, 1, n) + W.qft(n)) + ((rings(n, 6),) if n > 12 else ()):
        passes, _, text = K.Circuit(n, gates).plan(dtype)
        assert text.count(" stream") == passes
        assert passes <= K.Circuit(n, gates).plan(dtype, tile_qubits=12)[0]
