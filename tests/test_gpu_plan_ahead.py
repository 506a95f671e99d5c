"""Passes of at most 512 tiles fetch the plan ahead, larger ones do not: states
on both sides of that line, each form of pass (light, register ops, streamed),
and a plan longer than the lines that are fetched, against the oracle."""
import numpy as np
import pytest

import kate_amd as K
from kate_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu

KINDS = {"layered": lambda n: W.layered(n, 2, 3), "qft": W.qft, "brickwork": lambda n: W.brickwork(n, 4, 7)}


def _check(n, gates, dtype, tol, tp):
    print("plan ahead", n, len(gates), dtype, flush=True)
    want = O.simulate(n, gates, tp)
    with K.Simulator(K.Circuit(n, gates), dtype=dtype) as sim:
        for _ in range(2):
            sim.execute(tp)
            assert np.max(np.abs(sim.state() - want)) < tol


# an amplitude goes through fewer than 1000 roundings: 1e3 * 2^-53 and 2^-24
@pytest.mark.parametrize("dtype,tol", [("c128", 1.2e-13), ("c64", 6e-5)])
@pytest.mark.parametrize("n", [13, 20, 21, 22])
@pytest.mark.parametrize("kind", sorted(KINDS))
def test_both_sides_of_the_line(gpu, kind, n, dtype, tol):
    _check(n, KINDS[kind](n), dtype, tol, W.basis_input(n, 5) if kind == "qft" else None)


@pytest.mark.parametrize("dtype,tol", [("c128", 1.2e-13), ("c64", 6e-5)])
@pytest.mark.parametrize("n", [10, 12])
def test_plan_longer_than_its_fetch(gpu, n, dtype, tol):
    _check(n, W.brickwork(n, 60, 11), dtype, tol, None)
    _check(n, W.layered(n, 60, 11), dtype, tol, None)
