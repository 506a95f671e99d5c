"""The plan text without a device is the simulator's own plan: streamed passes,
matrix-core steps and tiles of small states are in it."""
import re

import numpy as np
import pytest

import kate_amd as K
from kate_amd import workloads as W


def dense(n, k, count=6):
    rng = np.random.default_rng(n + k)
    return [W.Gate(W.DENSE, tuple(int(q) for q in rng.choice(n, size=k, replace=False)), 0, W.haar_unitary(rng, 1 << k))
            for _ in range(count)]


def test_streamed_passes_are_described():
    passes, _, text = K.Circuit(25, W.qft(25)).plan("c128")
    assert passes <= 4 and text.count(" stream") == passes
    # a shape of the caller's keeps the register ops
    assert " stream" not in K.Circuit(25, W.qft(25)).plan("c128", tile_qubits=12)[2]


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("k", [4, 5, 6])
def test_matrix_steps_are_described(k, dtype, monkeypatch):
    monkeypatch.setenv("KATE_DESCRIBE_OPS", "1")
    c = K.Circuit(14, dense(14, k))
    assert c.plan(dtype)[2].count(" mfma ") == 6
    assert " mfma " not in c.plan(dtype, matrix5=False)[2]


@pytest.mark.parametrize("n,tile", [(3, 10), (10, 10), (11, 11), (12, 12)])
def test_small_tiles_are_described(n, tile):
    text = K.Circuit(n, W.layered(n, 4, 1)).plan("c128")[2]
    assert re.match(rf"nq_int=12 tile_bits={tile} ", text)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("kind,n", [("layered", 8), ("layered", 22), ("qft", 11), ("qft", 20), ("dense", 15),
                                    ("brickwork", 18)])
def test_text_is_the_simulators(gpu, kind, n, dtype):
    gates = {"layered": lambda: W.layered(n, 6, 1), "qft": lambda: W.qft(n), "dense": lambda: dense(n, 5),
             "brickwork": lambda: W.brickwork(n, 6, 1)}[kind]()
    c = K.Circuit(n, gates)
    with K.Simulator(c, dtype=dtype) as sim:
        assert sim.describe() == c.plan(dtype)[2]
