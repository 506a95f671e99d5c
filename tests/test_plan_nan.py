"""A gate entry that is NaN stays in the plan: the planner's rewritings of a gate
(Euler form, Kronecker factors) rebuild the gate and compare it with the
original, and a comparison with NaN has to fail."""
import re

import numpy as np
import pytest

import kate_amd as K
from kate_amd import workloads as W


def ops(gates, n, monkeypatch):
    monkeypatch.setenv("KATE_DESCRIBE_OPS", "1")
    return re.findall(r" (dense|kron|ekron|fkron):(\d+)", K.Circuit(n, gates).plan("c128", reorder=False)[2])


def haar(seed, dim):
    return W.haar_unitary(np.random.default_rng(seed), dim)


@pytest.mark.parametrize("entry", range(4))
def test_one_qubit_gate_keeps_nan(entry, monkeypatch):
    def gates(nan):
        out = [W.Gate(W.DENSE, (q,), 0, haar(q, 2)) for q in range(4)]
        if nan:
            out[1].mat.reshape(-1)[entry] = np.nan
        return out
    assert ops(gates(False), 4, monkeypatch)[0][0] == "ekron"
    assert [k for k, _ in ops(gates(True), 4, monkeypatch)] == ["kron"]


@pytest.mark.parametrize("entry", range(16))
def test_two_qubit_gate_keeps_nan(entry, monkeypatch):
    u = np.kron(haar(1, 2), haar(2, 2))
    assert ops([W.Gate(W.DENSE, (0, 1), 0, u)], 4, monkeypatch)[0][0] != "dense"
    u.reshape(-1)[entry] = np.nan
    (kind, mask), = ops([W.Gate(W.DENSE, (0, 1), 0, u)], 4, monkeypatch)
    assert kind == "dense" and bin(int(mask)).count("1") == 2
