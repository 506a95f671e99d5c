"""The work that programs built on kate_amd have it do, as measurable cases.

A case is one call sequence through the public classes (`Simulator`, `Batch`,
`Server`) on a circuit family and size taken from this repository's workloads
(`kate_amd/workloads.py`, `kate_amd/serving.py`, `bench.py`, the tests):

* ``listed()`` names the representative ones, ``draw()`` makes more of the
  same ranges;
* ``prepare()`` makes what a program has in hand before the call (the planned
  simulator, the captured batch, the running server), ``run()`` is one call;
* ``exact()`` computes the same outputs in 64 bits with plain torch.

Results of complex64 states are returned in 32 bits, the precision they
carry, and without Kate's proba_state: it is made of quotients of sums over all
amplitudes, and where such a sum nearly cancels, 32-bit amplitudes leave no
fixed number of its digits.
"""
import math

import numpy as np
import torch

import kate_amd as K
from kate_amd import workloads as W

# Circuit families:
#   layered    RX, RZ on every qubit then the CNOT ladder, per layer
#   brickwork  Haar 2-qubit brickwork with long-range layers
#   qft        Kate's QFT
#   mixed      every gate kind on random qubits, Haar dense gates of up to `k` qubits
#   dense      Haar dense gates of `k` qubits on random qubits
#   batch      many brickwork circuits of 10..`n` qubits in one captured launch
#   serve      requests (layered circuits and QFTs of 12..`n` qubits) through the server
_AMP = {"c128": 16, "c64": 8}


def listed():
    return [
        # The smallest calls: a variational loop on a few qubits that reads its
        # state back on every call.  Launches and latency.
        dict(name="small_10q_c128", kind="layered", n=10, depth=10, dtype="c128", input="zero", zs=4),
        # A laptop-sized circuit on the plain path (the 20-qubit, 10-layer parity circuit).
        dict(name="layered_20q_c128", kind="layered", n=20, depth=10, dtype="c128", input="zero", zs=8),
        # The headline: 30 qubits, depth 20, every pass over a 16 GiB state.
        dict(name="layered_30q_c128", kind="layered", n=30, depth=20, dtype="c128", input="zero", zs=8),
        # The complex64 form of it after Kate's gate fusion, with the Pauli terms of a small Hamiltonian.
        dict(name="fused_28q_c64", kind="layered", n=28, depth=20, dtype="c64", input="zero", fuse=5, zs=40),
        # Random-circuit sampling: dense 2-qubit gates, neighbours and long range.
        dict(name="brickwork_27q_c128", kind="brickwork", n=27, depth=24, dtype="c128", input="zero", zs=8),
        # The same compiled for 8 GPUs: its qubit swaps run as passes on this one.
        dict(name="swaps_28q_c64", kind="brickwork", n=28, depth=16, dtype="c64", input="zero", gpus=3, zs=40),
        # QFT of a product state: controlled phases, an input of the caller's.
        dict(name="qft_25q_c128", kind="qft", n=25, dtype="c128", input="product", zs=8),
        # An odd size with every gate kind (Toffoli, CRk, dense gates of 1..4 qubits).
        dict(name="mixed_23q_c64", kind="mixed", n=23, gates=300, k=4, dtype="c64", input="product", zs=40),
        # Wide dense gates, what fusing to 5 qubits makes of a deep circuit: both precisions.
        dict(name="dense5_26q_c128", kind="dense", n=26, gates=40, k=5, dtype="c128", input="zero", zs=8),
        dict(name="dense5_27q_c64", kind="dense", n=27, gates=60, k=5, dtype="c64", input="zero", zs=40),
        # Parameter sweeps: many small circuits at once, <Z> of every qubit.
        dict(name="batch_256_c64", kind="batch", n=20, count=256, dtype="c64"),
        # Serving: requests of 12..24 qubits in flight together, planned on arrival.
        dict(name="serve_24_c128", kind="serve", n=24, count=24, dtype="c128"),
    ]


def draw(rng):
    kind = rng.choice(("layered", "layered", "layered", "brickwork", "brickwork", "qft", "mixed", "dense", "batch",
                       "serve"))
    dtype = rng.choice(("c128", "c64"))
    if kind == "batch":
        count = int(round(math.exp(rng.uniform(math.log(16), math.log(256)))))
        return dict(kind=kind, n=rng.randint(13, 20), count=count, dtype=dtype)
    if kind == "serve":
        return dict(kind=kind, n=rng.randint(14, 24), count=rng.randint(3, 24), dtype=dtype)
    # state sizes spread over their logarithm
    top = {"layered": 29, "brickwork": 28, "qft": 28, "mixed": 24, "dense": 26}[kind]
    c = dict(kind=kind, n=rng.randint(6, top), dtype=dtype, input=rng.choice(("zero", "product")),
             zs=rng.randint(16, 48))
    if kind == "layered":
        c["depth"] = rng.randint(4, 24)
        if rng.random() < 0.4:
            c["fuse"] = rng.randint(2, 5)
    elif kind == "brickwork":
        c["depth"] = rng.randint(4, 24)
        if rng.random() < 0.3 and c["n"] >= 14:
            c["gpus"] = rng.randint(1, 3)
    elif kind == "mixed":
        c.update(gates=rng.randint(40, 300), k=rng.randint(2, 6), input="product")
    elif kind == "dense":
        c.update(gates=rng.randint(8, 40), k=rng.randint(2, 6))
        if c["k"] == 6:
            c["n"] = min(c["n"], 23)
    elif kind == "qft":
        c["input"] = "product"
    return c


# ---- inputs ------------------------------------------------------------------

def _gates(c, seed):
    n = c["n"]
    if c["kind"] == "layered":
        return W.layered(n, c["depth"], seed)
    if c["kind"] == "brickwork":
        return W.brickwork(n, c["depth"], seed)
    if c["kind"] == "qft":
        return W.qft(n)
    rng = np.random.default_rng(seed)
    if c["kind"] == "mixed":
        # a Haar gate on every qubit first, so that no qubit keeps a symmetric state
        first = [W.Gate(W.DENSE, (q,), 0, W.haar_unitary(rng, 2)) for q in range(n)]
        return first + W.random_mixed(n, c["gates"], seed, max_dense=c["k"])
    k = c["k"]
    out = []
    for u in W.haar_unitaries(rng, c["gates"], 1 << k):
        out.append(W.Gate(W.DENSE, tuple(int(q) for q in rng.choice(n, size=k, replace=False)), 0, u))
    return out


def _angles(n, seed):
    rng = np.random.default_rng([seed, 7])
    return np.stack([rng.uniform(0.1, 0.9, n), rng.uniform(0.0, 2 * math.pi, n)], axis=1)


def _masks(n, count, seed):
    return [int(m) for m in W.zstring_masks(n, count, seed)]


def _sizes(c, nmin):
    """A fixed number of qubits per circuit, spread evenly over the logarithm of
    the range and in mixed order."""
    k = c["count"]
    return [int(round(math.exp(math.log(nmin) + (i * 7 % k + 0.5) / k * math.log(c["n"] / nmin)))) for i in range(k)]


def _circuits(c, seed):
    """(n, gates) per circuit of a batch: Haar brickwork, depth 8..32."""
    rng = np.random.default_rng(seed)
    out = []
    for i, n in enumerate(_sizes(c, 10)):
        depth = 8 + i * 11 % 25
        u = iter(W.haar_unitaries(rng, depth * (n // 2), 4))
        out.append((n, [W.Gate(W.DENSE, (a, a + 1), 0, next(u)) for d in range(depth) for a in range(d % 2, n - 1, 2)]))
    return out


def _requests(c, seed):
    """(n, gates, masks, angles or None) per request: half layered circuits
    from |0...0>, half QFTs of product states."""
    out = []
    for i, n in enumerate(_sizes(c, 12)):
        s = seed * 1009 + i
        if i % 2 == 0:
            out.append((n, W.layered(n, 10 + i * 13 % 21, s), _masks(n, 8, s), None))
        else:
            out.append((n, W.qft(n), _masks(n, 8, s), _angles(n, s)))
    return out


# ---- the calls ----------------------------------------------------------------

class _DeviceState:
    """The simulator's state in HBM, for torch (no copy)."""

    def __init__(self, sim, n, dtype):
        self.sim = sim
        self.__cuda_array_interface__ = {"shape": (1 << n,), "typestr": "<c%d" % _AMP[dtype], "strides": None,
                                         "data": (sim.device_state(), False), "version": 2}


def prepare(case, seed):
    kind, dtype = case["kind"], case["dtype"]
    if kind == "batch":
        batch = K.Batch([K.Circuit(n, g) for n, g in _circuits(case, seed)], dtype=dtype)
        batch.capture()
        return {"kind": kind, "dtype": dtype, "batch": batch}
    if kind == "serve":
        reqs = [(K.Circuit(n, g), m, tp) for n, g, m, tp in _requests(case, seed)]
        server = K.Server(dtype=dtype, hbm_budget_bytes=8 << 30)
        return {"kind": kind, "dtype": dtype, "requests": reqs, "server": server}
    n = case["n"]
    c = K.Circuit(n, _gates(case, seed))
    if case.get("fuse"):
        c.schedule().fuse(case["fuse"])
    if case.get("gpus"):
        c.schedule().group(10).allocate(case["gpus"])
    return {"kind": kind, "dtype": dtype, "n": n, "sim": K.Simulator(c, dtype=dtype),
            "angles": _angles(n, seed) if case["input"] == "product" else None, "masks": _masks(n, case["zs"], seed)}


def _values(x, dtype):
    return np.asarray(x, dtype=np.float64 if dtype == "c128" else np.float32)


def run(state):
    dtype = state["dtype"]
    if state["kind"] == "batch":
        state["batch"].run()
        z, norms = state["batch"].expect_z()
        return {"z": _values(np.concatenate(z), dtype), "norms": _values(norms, dtype)}
    if state["kind"] == "serve":
        srv = state["server"]
        ids = [srv.submit(c, m, tp) for c, m, tp in state["requests"]]
        return {"z": _values(np.concatenate([srv.wait(i)[0] for i in ids]), dtype)}
    sim, n = state["sim"], state["n"]
    proba = sim.execute(state["angles"])
    z = sim.expect_z(state["masks"])
    # small states are read back, large ones stay in HBM for the next consumer
    amps = sim.state(real_order=False) if n < 16 else torch.as_tensor(_DeviceState(sim, n, dtype), device="cuda")
    out = {"z": _values(z, dtype), "state": amps}
    if dtype == "c128":
        out["proba"] = proba
    return out


# ---- what a call cannot do without -----------------------------------------------

def _gate_flops(n, gates):
    f = 0.0
    for g in gates:
        if g.id == W.DENSE:
            f += 8.0 * (1 << n) * (1 << len(g.qubits))
        elif g.id == W.H:
            f += 4.0 * (1 << n)
        elif g.id == W.CRK:
            f += 1.5 * (1 << n)
    return f


def work(case):
    amp = _AMP[case["dtype"]]
    if case["kind"] == "batch":
        circuits = _circuits(case, 1)
        return {"bytes": float(sum(amp << n for n, _ in circuits)),
                "flops": sum(_gate_flops(n, g) for n, g in circuits)}
    if case["kind"] == "serve":
        reqs = _requests(case, 1)
        return {"bytes": float(sum(amp << r[0] for r in reqs)), "flops": sum(_gate_flops(r[0], r[1]) for r in reqs)}
    # the finished state is written once
    return {"bytes": float(amp << case["n"]), "flops": _gate_flops(case["n"], _gates(case, 1))}


# ---- the same outputs in 64 bits, with plain torch ----------------------------------

def _split(v, n, qubits):
    """v with a dimension of its own for each of `qubits`; the dimension of each."""
    desc = sorted(qubits, reverse=True)
    shape, dims, hi = [], {}, n
    for q in desc:
        shape += [1 << (hi - 1 - q), 2]
        dims[q] = len(shape) - 1
        hi = q
    return v.view(shape + [1 << hi]), dims


def _apply(v, n, g):
    t, dims = _split(v, n, g.qubits)

    def at(**fixed):
        ix = [slice(None)] * t.dim()
        for name, val in fixed.items():
            ix[dims[g.qubits[int(name[1:])]]] = val
        return t[tuple(ix)]

    if g.id == W.CRK:
        at(q0=1, q1=1).mul_(complex(math.cos(2 * math.pi / 2 ** g.optarg), math.sin(2 * math.pi / 2 ** g.optarg)))
        return v
    if g.id in (W.CNOT, W.TOFFOLI):
        a, b = (at(q0=0, q1=1), at(q0=1, q1=1)) if g.id == W.CNOT else (at(q0=1, q1=1, q2=0), at(q0=1, q1=1, q2=1))
        keep = a.clone()
        a.copy_(b)
        b.copy_(keep)
        return v
    m = np.array([[1, 1], [1, -1]], dtype=np.complex128) / math.sqrt(2) if g.id == W.H else g.mat
    if len(g.qubits) == 1:
        a, b = at(q0=0), at(q0=1)
        if m[0, 1] == 0 and m[1, 0] == 0:
            a.mul_(complex(m[0, 0]))
            b.mul_(complex(m[1, 1]))
            return v
        new = a * complex(m[0, 0])
        new.add_(b, alpha=complex(m[0, 1]))
        b.mul_(complex(m[1, 1])).add_(a, alpha=complex(m[1, 0]))
        a.copy_(new)
        return v
    front = [dims[q] for q in reversed(g.qubits)]
    order = front + [d for d in range(t.dim()) if d not in front]
    p = t.permute(order)
    r = torch.from_numpy(np.ascontiguousarray(m)).to(v.device) @ p.reshape(1 << len(front), -1)
    back = [order.index(d) for d in range(t.dim())]
    return r.view(p.shape).permute(back).reshape(-1)


def _input(n, angles, dev):
    v = torch.ones(1, dtype=torch.complex128, device=dev)
    for q in range(n):
        if angles is None:
            f = [1.0, 0.0]
        else:
            th, ph = angles[q]
            f = [math.cos(th * math.pi / 2), complex(math.cos(ph), math.sin(ph)) * math.sin(th * math.pi / 2)]
        v = torch.kron(torch.tensor(f, dtype=torch.complex128, device=dev), v)
    return v


def _simulate(n, gates, angles, dev):
    v = _input(n, angles, dev)
    for g in gates:
        v = _apply(v, n, g)
    return v


def _zstrings(v, n, masks):
    p = v.real.square().add_(v.imag.square())
    out = []
    for m in masks:
        t = p
        for q in range(n - 1, -1, -1):
            t = t.view(2, -1)
            t = t[0] - t[1] if (m >> q) & 1 else t[0] + t[1]
        out.append(t.reshape(()))
    return (torch.stack(out) / p.sum()).cpu().numpy(), float(p.sum())


def _proba(v, n):
    """Kate's proba_state: (theta, phi) of each qubit from the sums of the
    amplitudes in which it is 0 and 1."""
    total = v.sum()
    out = np.zeros((n, 2))
    for q in range(n):
        s1 = v.view(-1, 2, 1 << q)[:, 1].sum()
        den = math.sqrt(2.0) ** n
        a0, a1 = complex(total - s1) / den, complex(s1) / den
        if abs(a0) < 1e-13:
            out[q] = 1, 0
        elif abs(a1) >= 1e-14:
            r = a1 / a0
            out[q] = math.atan(abs(r)) / (math.pi / 2), math.atan(r.imag / r.real)
    return out


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if case["kind"] == "batch":
        z, norms = [], []
        for n, gates in _circuits(case, seed):
            zs, norm = _zstrings(_simulate(n, gates, None, dev), n, [1 << q for q in range(n)])
            z.append(zs)
            norms.append(norm)
        return {"z": np.concatenate(z), "norms": np.array(norms)}
    if case["kind"] == "serve":
        z = [_zstrings(_simulate(n, g, tp, dev), n, m)[0] for n, g, m, tp in _requests(case, seed)]
        return {"z": np.concatenate(z)}
    n = case["n"]
    if n > 28:
        return None
    v = _simulate(n, _gates(case, seed), _angles(n, seed) if case["input"] == "product" else None, dev)
    z, _ = _zstrings(v, n, _masks(n, case["zs"], seed))
    # a program with swaps leaves its state in another qubit order
    out = {"z": z, "state": None if case.get("gpus") else v}
    if case["dtype"] == "c128":
        out["proba"] = _proba(v, n)
    return out
