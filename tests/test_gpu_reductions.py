"""The reductions (Z strings, Kate's proba_state, <Z> of a batch) against
plain sums over the same amplitudes, at the sizes where their split changes:
one chunk of 4096 amplitudes, one chunk per workgroup, more chunks than
workgroups, and mask counts around one launch's limit."""
import numpy as np
import pytest

import kate_amd as K
from kate_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def random_state(n, dtype, seed):
    rng = np.random.default_rng(seed)
    st = rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)
    return (st / np.linalg.norm(st)).astype(np.complex128 if dtype == "c128" else np.complex64)


def z_of(st, n, masks):
    p = st.real.astype(np.float64) ** 2 + st.imag.astype(np.float64) ** 2
    out = []
    for m in masks:
        t = p
        for q in range(n - 1, -1, -1):
            t = t.reshape(2, -1)
            t = t[0] - t[1] if (int(m) >> q) & 1 else t[0] + t[1]
        out.append(float(t.reshape(())))
    return np.array(out) / p.sum()


# FP64 sums of n levels of additions over probabilities that add up to 1: the
# error is below (n + 16) eps, 1e-14 at these sizes; 16 + 256 terms are added
# one after the other at the largest (6e-14).
@pytest.mark.parametrize("n,dtype,count", [(3, "c128", 5), (12, "c64", 64), (13, "c128", 1), (14, "c64", 65),
                                           (23, "c64", 63), (24, "c128", 130), (25, "c64", 7)])
def test_z_strings(n, dtype, count):
    st = random_state(n, dtype, n)
    masks = [int(m) for m in W.zstring_masks(n, count, n)]
    masks[0] = 1 << (n - 1)
    masks[-1] = 1
    with K.Simulator(K.Circuit(n, [W.Gate(W.H, (0,))]), dtype=dtype) as sim:
        sim.write_state(st)
        got = sim.expect_z(masks)
        assert np.max(np.abs(got - z_of(st, n, masks))) < 1e-13
        assert abs(sim.norm() - float(np.sum(np.abs(st.astype(np.complex128)) ** 2))) < 1e-13


# theta and phi are arctangents of quotients of the sums; random sums are of
# order 1 with errors of 1e-14 at most, so that the angles hold to 1e-9 even
# where a quotient is a thousand times worse conditioned.
@pytest.mark.parametrize("n,dtype", [(5, "c128"), (12, "c64"), (13, "c128"), (16, "c64"), (23, "c128"), (24, "c64")])
def test_proba_sums(n, dtype):
    st = random_state(n, dtype, 100 + n)
    with K.Simulator(K.Circuit(n, [W.Gate(W.H, (0,))]), dtype=dtype) as sim:
        sim.write_state(st)
        got = sim.measure_proba()
    ref = O.measure(n, st.astype(np.complex128))
    assert np.max(np.abs(got - ref)) < 1e-9


# The batch's sums against the simulator's on the same circuits: one block of
# 2^14 amplitudes, less than one, and several.  Both are FP64 sums over the
# same kind of state; the states agree to their own rounding (1e-12 for
# complex128, as everywhere in these tests).
@pytest.mark.parametrize("tile", [10, 12])
def test_batch_z_blocks(tile):
    sizes = [4, 10, 13, 14, 15, 17]
    circuits = [K.Circuit(n, W.layered(n, 3, n)) for n in sizes]
    with K.Batch(circuits, dtype="c128", tile_qubits=tile) as b:
        b.run()
        z, norms = b.expect_z()
    for n, c, zc, norm in zip(sizes, circuits, z, norms):
        with K.Simulator(c) as sim:
            sim.execute()
            assert np.max(np.abs(zc - sim.expect_z([1 << q for q in range(n)]))) < 1e-12
        assert abs(norm - 1) < 1e-12
