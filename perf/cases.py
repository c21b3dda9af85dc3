"""The workloads this engine is timed on.

Each case is one pass of a program that holds a register, a compiled gate
sequence, a batch of instances or a network, and calls the engine's public
entry points on it: single gates, gate lists (plain and fused), recorded
sequences, the Fourier transform, sampling, Pauli-string expectations, batched
QAOA and VQE energies, and the surrogate network.

Values that a complex64 register or a complex64 batch computes are returned in
single precision, the precision that they carry. States are returned where a
program of that size reads them; larger registers return what such a program
reads instead: sampled outcomes and expectation values.
"""
import ctypes
import math

import numpy as np
import torch

from qcsim_amd import QuantumFourierTransform, QubitRegister, lib
from qcsim_amd import gates as G
from qcsim_amd._lib import check
from qcsim_amd.learned import Surrogate
from qcsim_amd.qaoa import IsingInstance, QaoaBatch
from qcsim_amd.vqe import VqeBatch

_PF = ctypes.POINTER(ctypes.c_float)
_SIZES = (12, 14, 16, 18, 20, 22)


def listed():
    return [
        # a small program: gates of every family applied one call at a time, a
        # mid-circuit measurement, the state read back
        {"name": "eager_10q", "kind": "eager", "n": 10, "precision": "c128", "gates": 80},
        # recorded gates replayed on a register of ordinary size, the state read back
        {"name": "replay_16q", "kind": "replay", "n": 16, "precision": "c128", "gates": 600, "width": 0},
        # the 20-qubit workload: 40 layers of Haar U(2) and CNOT / CZ / controlled
        # U(2) pairs, a Fourier transform, 1024 samples
        {"name": "layers_20q", "kind": "layers", "n": 20, "precision": "c128", "layers": 40, "width": 0},
        # the same kind of circuit through the fusion pass, on a register with an odd number of qubits
        {"name": "layers_25q_fused", "kind": "layers", "n": 25, "precision": "c128", "layers": 16, "width": 5},
        # time evolution of an Ising chain in complex64, fused
        {"name": "trotter_27q_c64", "kind": "trotter", "n": 27, "precision": "c64", "steps": 6, "width": 5},
        # the headline sweep: one U(2) call per target on 16 GiB
        {"name": "sweep_30q", "kind": "sweep", "n": 30, "precision": "c128"},
        # phase estimation's two transforms, inverse and forward, on 8 GiB
        {"name": "qft_29q", "kind": "qft", "n": 29, "precision": "c128", "shots": 256},
        # the energy terms of a Heisenberg chain
        {"name": "heisenberg_26q", "kind": "heisenberg", "n": 26, "precision": "c128"},
        # one evaluation of many uneven QAOA instances
        {"name": "qaoa_256", "kind": "qaoa", "instances": 256, "smallest": 12, "largest": 22, "p": 4},
        # one gradient's evaluations of a batch of VQE instances
        {"name": "vqe_1024", "kind": "vqe", "instances": 1024, "smallest": 4, "largest": 12, "terms": 24, "depth": 2},
        # scoring 65536 candidate angle sets
        {"name": "predict_65536", "kind": "predict", "rows": 65536, "inputs": 17, "hidden": 256, "layers": 3},
        # training the surrogate
        {"name": "train_131072", "kind": "train", "rows": 131072, "inputs": 17, "hidden": 256, "layers": 3,
         "batch": 4096, "epochs": 1},
    ]


def _spread(rng, lo, hi):
    """A whole number between lo and hi, even over the logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5))))))


def draw(rng):
    kind = rng.choice(("eager", "replay", "layers", "trotter", "sweep", "qft", "heisenberg", "qaoa", "vqe", "predict",
                       "train"))
    prec = rng.choice(("c128", "c64"))
    if kind == "eager":
        return {"kind": kind, "n": rng.randint(3, 15), "precision": prec, "gates": _spread(rng, 20, 200)}
    if kind == "replay":
        return {"kind": kind, "n": rng.randint(6, 20), "precision": prec, "gates": _spread(rng, 50, 800),
                "width": rng.choice((0, 0, 4, 5))}
    if kind == "layers":
        n = rng.randint(14, 25)
        return {"kind": kind, "n": n, "precision": "c128", "layers": rng.randint(4, 40 if n < 23 else 14),
                "width": rng.choice((0, 4, 5))}
    if kind == "trotter":
        n = rng.randint(12, 27)
        return {"kind": kind, "n": n, "precision": prec, "steps": rng.randint(2, 12 if n < 25 else 5),
                "width": rng.choice((0, 4, 5) if n < 25 else (4, 5))}
    if kind == "sweep":
        return {"kind": kind, "n": rng.randint(20, 30), "precision": prec}
    if kind == "qft":
        return {"kind": kind, "n": rng.randint(8, 29), "precision": "c128", "shots": _spread(rng, 2, 4096)}
    if kind == "heisenberg":
        return {"kind": kind, "n": rng.randint(6, 27), "precision": prec}
    if kind == "qaoa":
        lo = rng.randrange(0, len(_SIZES))
        return {"kind": kind, "instances": _spread(rng, 1, 256), "smallest": _SIZES[lo],
                "largest": _SIZES[rng.randrange(lo, len(_SIZES))], "p": rng.randint(1, 4)}
    if kind == "vqe":
        lo = rng.randint(1, 12)
        return {"kind": kind, "instances": _spread(rng, 8, 1024), "smallest": lo, "largest": rng.randint(lo, 12),
                "terms": _spread(rng, 2, 48), "depth": rng.randint(1, 4)}
    if kind == "predict":
        return {"kind": kind, "rows": _spread(rng, 1, 100000), "inputs": 9 + 2 * rng.randint(1, 6),
                "hidden": rng.choice((64, 96, 128, 200, 256)), "layers": rng.randint(1, 4)}
    batch = _spread(rng, 200, 4096)
    return {"kind": "train", "rows": batch * rng.randint(2, 16) + rng.randint(0, batch - 1),
            "inputs": 9 + 2 * rng.randint(1, 4), "hidden": rng.choice((64, 96, 128, 256)), "layers": rng.randint(1, 3),
            "batch": batch, "epochs": rng.randint(1, 2)}


# ---- gates: (name, qubits, argument), the first qubit is the target -------------------

_S2 = 1 / math.sqrt(2)
_X = np.array([[0, 1], [1, 0]], dtype=complex)
_ONE = ("u", "h", "x", "t", "rx", "ry", "rz")
_TWO = ("cx", "cz", "cp", "cu", "swap", "iswap")
_THREE = ("ccx", "ccz", "cswap")


def _haar(rng):
    z = rng.standard_normal((2, 2)) + 1j * rng.standard_normal((2, 2))
    q, r = np.linalg.qr(z)
    return q * (np.diagonal(r) / np.abs(np.diagonal(r)))


def _gate(op):
    """The engine's gate object."""
    name, _, a = op
    if name == "u":
        return G.SingleQubitGate(a)
    if name == "cu":
        g = G.TwoQubitsControlledGate()
        g.SetOperation(a)
        return g
    if name in ("rx", "ry", "rz", "cp"):
        return {"rx": G.RxGate, "ry": G.RyGate, "rz": G.RzGate, "cp": G.ControlledPhaseShiftGate}[name](a)
    return {"h": G.HadamardGate, "x": G.PauliXGate, "t": G.TGate, "cx": G.CNOTGate, "cz": G.ControlledZGate,
            "swap": G.SwapGate, "iswap": G.iSwapGate, "ccx": G.ToffoliGate, "ccz": G.CCZGate,
            "cswap": G.FredkinGate}[name]()


def _matrix(op):
    """The gate's matrix from its definition: bit i of an index is the gate's qubit i."""
    name, _, a = op
    if name == "rx":
        c, s = math.cos(a / 2), math.sin(a / 2)
        return np.array([[c, -1j * s], [-1j * s, c]])
    if name == "ry":
        c, s = math.cos(a / 2), math.sin(a / 2)
        return np.array([[c, -s], [s, c]], dtype=complex)
    if name == "rz":
        return np.diag([np.exp(-0.5j * a), np.exp(0.5j * a)])
    small = {"u": a, "h": np.array([[_S2, _S2], [_S2, -_S2]]), "x": _X, "t": np.diag([1, np.exp(0.25j * math.pi)])}
    if name in small:
        return np.asarray(small[name], dtype=complex)
    m = np.eye(8 if name in _THREE else 4, dtype=complex)
    if name in ("cx", "cu"):
        m[2:, 2:] = _X if name == "cx" else a
    elif name in ("cz", "cp"):
        m[3, 3] = -1 if name == "cz" else np.exp(1j * a)
    elif name in ("swap", "iswap"):
        m[1, 1] = m[2, 2] = 0
        m[1, 2] = m[2, 1] = 1 if name == "swap" else 1j
    elif name == "ccx":
        m[6:, 6:] = _X
    elif name == "ccz":
        m[7, 7] = -1
    else:
        m[5, 5] = m[6, 6] = 0
        m[5, 6] = m[6, 5] = 1
    return m


def _mixed(n, count, rng):
    """Gates of every family on random qubits."""
    ops = []
    for _ in range(count):
        r = rng.random()
        family = _ONE if r < 0.6 or n < 2 else _TWO if r < 0.93 or n < 3 else _THREE
        name = family[rng.integers(len(family))]
        k = 1 if family is _ONE else 2 if family is _TWO else 3
        a = _haar(rng) if name in ("u", "cu") else float(rng.uniform(0, 2 * math.pi))
        ops.append((name, tuple(int(q) for q in rng.permutation(n)[:k]), a))
    return ops


def _layers(n, layers, rng):
    """Layers of a Haar U(2) on every qubit, then CNOT, CZ or controlled U(2) on a random pairing."""
    ops = []
    for _ in range(layers):
        ops += [("u", (q,), _haar(rng)) for q in range(n)]
        perm = [int(q) for q in rng.permutation(n)]
        for a, b in zip(perm[0::2], perm[1::2]):
            name = ("cx", "cz", "cu")[rng.integers(3)]
            ops.append((name, (a, b), _haar(rng) if name == "cu" else 0.0))
    return ops


def _trotter(n, steps, rng):
    """First-order steps of an Ising chain in a transverse field from a tilted product state."""
    J, hx = rng.uniform(0.5, 1.0, n), rng.uniform(0.3, 0.8, n)
    ops = [("ry", (q,), float(rng.uniform(0.2, 0.9))) for q in range(n)]
    for _ in range(steps):
        for q in range(n - 1):
            ops += [("cx", (q + 1, q), 0.0), ("rz", (q + 1,), float(0.2 * J[q])), ("cx", (q + 1, q), 0.0)]
        ops += [("rx", (q,), float(0.2 * hx[q])) for q in range(n)]
    return ops


def _entangled(n, rng):
    """A product of random qubit states, then two rows of CNOTs between neighbours."""
    ops = [("u", (q,), _haar(rng)) for q in range(n)]
    ops += [("cx", (q + 1, q), 0.0) for start in (0, 1) for q in range(start, n - 1, 2)]
    return ops + [("u", (q,), _haar(rng)) for q in range(n)]


def _pairs(ops):
    """The gate list as QubitRegister.apply_circuit takes it."""
    return [(_gate(op), list(op[1])) for op in ops]


def _z_terms(n):
    return np.zeros(n, dtype=np.uint64), np.array([1 << q for q in range(n)], dtype=np.uint64)


def _chain_terms(n):
    """Masks of the terms of a Heisenberg chain in a field: XX, YY and ZZ of each bond, Z of each site."""
    x, z = [], []
    for q in range(n - 1):
        b = 3 << q
        x += [b, b, 0]
        z += [0, b, b]
    return np.array(x + [0] * n, dtype=np.uint64), np.array(z + [1 << q for q in range(n)], dtype=np.uint64)


def _phases(n, rng):
    """The phases of a register that holds a Fourier state, each a little off."""
    phi = rng.random()
    return [2 * math.pi * ((phi * 2**q) % 1.0) + float(rng.normal(0, 0.15)) for q in range(n)]


def _ising(n, rng):
    """A weighted Ising model on a random 3-regular graph."""
    while True:
        stubs = rng.permutation(np.repeat(np.arange(n), 3)).reshape(-1, 2)
        edges = {(int(min(e)), int(max(e))) for e in stubs if e[0] != e[1]}
        if len(edges) == 3 * n // 2:
            break
    edges = sorted(edges)
    return IsingInstance(n, edges, rng.normal(0, 1, len(edges)), rng.normal(0, 0.5, n))


def _qaoa(case, rng):
    sizes = [s for s in _SIZES if case["smallest"] <= s <= case["largest"]]
    insts = [_ising(sizes[i % len(sizes)], rng) for i in range(case["instances"])]
    shape = (case["instances"], case["p"])
    return insts, rng.uniform(0, math.pi, shape), rng.uniform(0, math.pi, shape)


def _vqe(case, rng):
    insts, params = [], []
    for _ in range(case["instances"]):
        n = int(rng.integers(case["smallest"], case["largest"] + 1))
        full = (1 << n) - 1
        xs = [0 if k % 4 == 0 else int(v) for k, v in enumerate(rng.integers(0, 1 << n, size=case["terms"]))]
        zs = [int(v) | (full & ~x) for v, x in zip(rng.integers(0, 1 << n, size=case["terms"]), xs)]
        insts.append((n, (xs, zs, [float(v) for v in rng.normal(size=case["terms"])])))
        params.append(rng.uniform(0, math.pi, size=2 * n * case["depth"]))
    return insts, params


def _network(case, rng):
    """Weights and biases, flat, as the engine lays them out, and the widths."""
    dims = [case["inputs"]] + [case["hidden"]] * case["layers"] + [1]
    parts = []
    for a, b in zip(dims[:-1], dims[1:]):
        lim = math.sqrt(6 / a)
        parts += [rng.uniform(-lim, lim, a * b), rng.normal(0, 0.05, b)]
    return dims, np.concatenate(parts).astype(np.float32)


def _features(rows, inputs, rng):
    """Instance statistics and angles over pi, as the surrogate's rows hold them."""
    x = rng.random((rows, inputs))
    x[:, : min(9, inputs)] += rng.normal(0, 0.5, min(9, inputs))
    return x.astype(np.float32)


# ---- what a program has in hand before the call ------------------------------------------


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind, s = case["kind"], {"case": case}
    if "precision" in case:
        s["reg"] = QubitRegister(case["n"], precision=case["precision"])
    n = case.get("n", 0)
    if kind == "eager":
        s["ops"] = [(g, q) for g, q in _pairs(_mixed(n, case["gates"], rng))]
        s["measured"], s["u"] = int(rng.integers(n)), float(rng.random())
    elif kind == "replay":
        s["program"] = s["reg"].compile_program(_pairs(_mixed(n, case["gates"], rng)), fuse_width=case["width"])
    elif kind == "layers":
        s["ops"], s["u"], s["terms"] = _pairs(_layers(n, case["layers"], rng)), rng.random(1024), _z_terms(n)
        s["qft"] = QuantumFourierTransform(n)
    elif kind == "trotter":
        s["ops"], s["terms"] = _pairs(_trotter(n, case["steps"], rng)), _z_terms(n)
    elif kind == "sweep":
        s["ops"], s["terms"] = [G.SingleQubitGate(_haar(rng)) for _ in range(n)], _z_terms(n)
    elif kind == "qft":
        for q, t in enumerate(_phases(n, rng)):
            s["reg"].ApplyGate(G.HadamardGate(), q)
            s["reg"].ApplyGate(G.PhaseShiftGate(t), q)
        s["u"], s["qft"] = rng.random(case["shots"]), QuantumFourierTransform(n)
        s["terms"] = tuple(t[-4:] for t in _z_terms(n))
    elif kind == "heisenberg":
        for g, q in _pairs(_entangled(n, rng)):
            s["reg"].ApplyGate(g, *q)
        s["terms"] = _chain_terms(n)
    elif kind == "qaoa":
        insts, s["gamma"], s["beta"] = _qaoa(case, rng)
        s["batch"] = QaoaBatch(insts, case["p"])
    elif kind == "vqe":
        insts, s["params"] = _vqe(case, rng)
        s["batch"] = VqeBatch(insts)
    else:
        dims, w = _network(case, rng)
        s["net"], s["w"] = Surrogate(case["inputs"], case["hidden"], case["layers"]), w
        check(lib().qcs_mlp_set_params(s["net"]._h, w.ctypes.data_as(_PF)))
        s["x"] = _features(case["rows"], case["inputs"], rng)
        if kind == "train":
            s["y"] = (np.sin(3 * s["x"][:, 0]) + 0.3 * s["x"][:, -1] + 0.1 * rng.standard_normal(case["rows"])).astype(
                np.float32)
    if "reg" in s:
        s["reg"].synchronize()
    return s


# ---- one pass -------------------------------------------------------------------------------


def _held(case, v):
    """Values in the precision of the register they come from."""
    if case["precision"] == "c128":
        return v
    return v.astype(np.complex64 if np.iscomplexobj(v) else np.float32)


def run(s):
    case, reg = s["case"], s.get("reg")
    kind = case["kind"]
    if kind == "eager":
        reg.Reset()
        half = len(s["ops"]) * 3 // 4
        for g, q in s["ops"][:half]:
            reg.ApplyGate(g, *q)
        bit = reg.MeasureQubit(s["measured"], u=s["u"])
        for g, q in s["ops"][half:]:
            reg.ApplyGate(g, *q)
        return {"bit": bit, "state": _held(case, reg.getRegisterStorage())}
    if kind == "replay":
        reg.Reset()
        s["program"].run()
        return {"state": _held(case, reg.getRegisterStorage())}
    if kind == "layers":
        reg.Reset()
        reg.apply_circuit(s["ops"], fuse_width=case["width"])
        z = reg.pauli_expectation(*s["terms"])
        s["qft"].QFT(reg)
        return {"z": z, "outcomes": reg.sample(s["u"])}
    if kind == "trotter":
        reg.Reset()
        reg.apply_circuit(s["ops"], fuse_width=case["width"])
        return {"z": _held(case, reg.pauli_expectation(*s["terms"]))}
    if kind == "sweep":
        reg.Reset()
        for q, g in enumerate(s["ops"]):
            reg.ApplyGate(g, q)
        return {"z": _held(case, reg.pauli_expectation(*s["terms"]))}
    if kind == "qft":
        s["qft"].IQFT(reg)
        outcomes, z = reg.sample(s["u"]), reg.pauli_expectation(*s["terms"])
        s["qft"].QFT(reg)
        return {"outcomes": outcomes, "z": z}
    if kind == "heisenberg":
        return {"terms": _held(case, reg.pauli_expectation(*s["terms"]))}
    if kind == "qaoa":  # complex64 states
        return {"energy": s["batch"].evaluate(s["gamma"], s["beta"]).astype(np.float32)}
    if kind == "vqe":
        return {"energy": s["batch"].evaluate(s["params"])}
    if kind == "predict":
        return {"y": s["net"].predict(s["x"])}
    losses = s["net"].train(s["x"], s["y"], batch=case["batch"], epochs=case["epochs"])
    w = np.empty_like(s["w"])
    check(lib().qcs_mlp_get_params(s["net"]._h, w.ctypes.data_as(_PF)))
    return {"losses": losses, "params": w}


# ---- what a pass cannot do without -------------------------------------------------------------

_FLOPS = {"u": 14, "h": 4, "rx": 8, "ry": 6, "rz": 6, "t": 3, "cu": 7, "cp": 1.5, "cz": 0.25, "ccz": 0.125}


def work(case):
    """Bytes and floating-point operations: registers written and read once, each single call's register read and
    written; gates by the complex products their matrices need."""
    kind, rng = case["kind"], np.random.default_rng(0)
    if "n" in case:
        n = case["n"]
        state = float((16 if case["precision"] == "c128" else 8) << n)
        amps = float(1 << n)
        gate_flops = lambda ops: amps * sum(_FLOPS.get(op[0], 0) for op in ops)  # noqa: E731
        if kind == "eager":
            return {"bytes": 2 * state * case["gates"], "flops": gate_flops(_mixed(n, case["gates"], rng))}
        if kind == "replay":
            return {"bytes": 2 * state, "flops": gate_flops(_mixed(n, case["gates"], rng))}
        if kind == "layers":
            return {"bytes": 4 * state, "flops": gate_flops(_layers(n, case["layers"], rng)) + 5 * n * amps}
        if kind == "trotter":
            return {"bytes": 2 * state, "flops": gate_flops(_trotter(n, case["steps"], rng))}
        if kind == "sweep":
            return {"bytes": 2 * state * n, "flops": 14 * amps * n}
        if kind == "qft":
            return {"bytes": 5 * state, "flops": 10 * n * amps}
        return {"bytes": state, "flops": 4 * amps * len(_chain_terms(n)[0])}
    if kind == "qaoa":
        sizes = [s for s in _SIZES if case["smallest"] <= s <= case["largest"]]
        sizes = [sizes[i % len(sizes)] for i in range(case["instances"])]
        return {"bytes": sum(16.0 * 2**n for n in sizes),
                "flops": sum((case["p"] * (8.0 * n + 6) + 4) * 2**n for n in sizes)}
    if kind == "vqe":
        sizes = [n for n, _ in _vqe(case, rng)[0]]
        return {"bytes": sum(24.0 * case["terms"] + 16 * n * case["depth"] + 8 for n in sizes),
                "flops": sum((20.0 * n * case["depth"] + 3 * case["terms"]) * 2**n for n in sizes)}
    i, h, k = case["inputs"], case["hidden"], case["layers"]
    weights = i * h + (k - 1) * h * h + h
    if kind == "predict":
        return {"bytes": 4.0 * case["rows"] * (i + 1) + 4 * weights, "flops": 2.0 * case["rows"] * weights}
    rows = case["rows"] // case["batch"] * case["batch"] * case["epochs"]
    return {"bytes": 4.0 * rows * (i + 1) + 8 * weights, "flops": 6.0 * rows * weights}


# ---- the same results in 64 bits ------------------------------------------------------------------


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _zero_state(n):
    psi = torch.zeros(1 << n, dtype=torch.complex128, device=_device())
    psi[0] = 1
    return psi


def _apply(psi, ops):
    n = psi.numel().bit_length() - 1
    for op in ops:
        m, qubits = _matrix(op), op[1]
        order = sorted(range(len(qubits)), key=lambda i: -qubits[i])
        shape, above = [], n
        for i in order:
            shape += [1 << (above - 1 - qubits[i]), 2]
            above = qubits[i]
        v = psi.view(shape + [1 << above])

        def at(local):
            idx = [slice(None)] * (2 * len(qubits) + 1)
            for j, i in enumerate(order):
                idx[2 * j + 1] = (local >> i) & 1
            return tuple(idx)

        rows = [r for r in range(len(m)) if np.any(m[r] != np.eye(len(m))[r])]
        new = []
        for r in rows:
            acc = None
            for c in np.nonzero(m[r])[0]:
                part = v[at(int(c))] * complex(m[r, c])
                acc = part if acc is None else acc.add_(part)
            new.append(acc)
        for r, x in zip(rows, new):
            v[at(r)] = x
    return psi


def _expect(psi, xs, zs):
    """<psi|P|psi> of the strings i^|x&z| X^x Z^z."""
    out, step = [], min(psi.numel(), 1 << 24)
    groups = {}
    for t, (x, z) in enumerate(zip(xs, zs)):
        groups.setdefault(int(x), []).append((t, int(z)))
    out = np.zeros(len(xs))
    for x, terms in groups.items():
        for start in range(0, psi.numel(), step):
            i = torch.arange(start, start + step, device=psi.device)
            a = psi[i ^ x].conj() * psi[start:start + step]  # conj(psi[i ^ x]) psi[i], which Z^z signs by i
            for t, z in terms:
                par = i & z
                for k in (16, 8, 4, 2, 1):
                    par = par ^ (par >> k)
                v = torch.sum(a * (1 - 2 * (par & 1)))
                out[t] += float((v * 1j ** (bin(x & z).count("1") % 4)).real)
    return out


def _qaoa_exact(inst, gamma, beta):
    n = inst.n
    i = torch.arange(1 << n, device=_device())
    z = [1.0 - 2.0 * ((i >> q) & 1).double() for q in range(n)]
    zz = torch.zeros(1 << n, dtype=torch.float64, device=_device())
    for (a, b), J in zip(inst.edges, inst.J):
        zz += J * z[a] * z[b]
    hz = sum(h * z[q] for q, h in enumerate(inst.h))
    psi = torch.full((1 << n,), 2.0 ** (-n / 2), dtype=torch.complex128, device=_device())
    for g, b in zip(gamma, beta):
        psi = psi * torch.exp(-1j * g * (zz + hz / 2))
        psi = _apply(psi, [("rx", (q,), 2 * float(b)) for q in range(n)])
    return float(-(psi.abs().square() * (zz + hz)).sum())


def _ansatz(n, params):
    """Ry / Rz layers and alternating CNOT ladders."""
    ops, pos, flip = [], 0, False
    while pos + 1 < len(params):
        if pos:
            if flip:
                ops += [("cx", (q - 1, q), 0.0) for q in range(n - 1, 0, -1)] + ([("cx", (n - 1, 0), 0.0)] if n > 2 else [])
            else:
                ops += [("cx", (q + 1, q), 0.0) for q in range(n - 1)] + ([("cx", (0, n - 1), 0.0)] if n > 2 else [])
            flip = not flip
        for q in range(n):
            ops += [("ry", (q,), float(params[pos])), ("rz", (q,), float(params[pos + 1]))]
            pos += 2
    return ops


def _vqe_exact(n, terms, params):
    i = np.arange(1 << n)
    psi = _apply(torch.zeros(1 << n, dtype=torch.complex128).index_fill_(0, torch.tensor([0]), 1), _ansatz(n, params))
    psi = psi.numpy()
    e = 0.0
    for x, z, c in zip(*terms):
        sign = 1 - 2.0 * (np.bitwise_count((i & z).astype(np.uint64)) & 1)
        e += c * float((np.vdot(psi[i ^ x], psi * sign) * 1j ** (bin(x & z).count("1") % 4)).real)
    return e


def _round_bf16(x):
    return x.float().bfloat16().double()


def exact(case, seed):
    rng = np.random.default_rng(seed)
    kind, n = case["kind"], case.get("n", 0)
    if kind == "eager":
        ops = _mixed(n, case["gates"], rng)
        q, u = int(rng.integers(n)), float(rng.random())
        half = len(ops) * 3 // 4
        psi = _apply(_zero_state(n), ops[:half])
        p = psi.abs().square()
        first = torch.nonzero(torch.cumsum(p, 0) >= 1 - u)  # the sampled state's value of the qubit
        bit = (int(first[0]) if len(first) else 0) >> q & 1
        keep = ((torch.arange(1 << n, device=psi.device) >> q) & 1) == bit
        psi = torch.where(keep, psi, 0) / math.sqrt(float(p[keep].sum()))
        return {"bit": None, "state": _apply(psi, ops[half:])}
    if kind == "replay":
        return {"state": _apply(_zero_state(n), _mixed(n, case["gates"], rng))}
    if kind == "layers":
        return {"z": _expect(_apply(_zero_state(n), _layers(n, case["layers"], rng)), *_z_terms(n)), "outcomes": None}
    if kind == "trotter":
        return {"z": _expect(_apply(_zero_state(n), _trotter(n, case["steps"], rng)), *_z_terms(n))}
    if kind == "sweep":
        u = [_haar(rng) for _ in range(n)]
        return {"z": np.array([abs(m[0, 0]) ** 2 - abs(m[1, 0]) ** 2 for m in u])}
    if kind == "qft":
        ops = []
        for q, t in enumerate(_phases(n, rng)):
            ops += [("h", (q,), 0.0), ("u", (q,), np.diag([1, np.exp(1j * t)]))]
        psi = torch.fft.fft(_apply(_zero_state(n), ops), norm="ortho")
        return {"outcomes": None, "z": _expect(psi, *(t[-4:] for t in _z_terms(n)))}
    if kind == "heisenberg":
        return {"terms": _expect(_apply(_zero_state(n), _entangled(n, rng)), *_chain_terms(n))}
    if kind == "qaoa":
        insts, gamma, beta = _qaoa(case, rng)
        return {"energy": np.array([_qaoa_exact(*a) for a in zip(insts, gamma, beta)])}
    if kind == "vqe":
        insts, params = _vqe(case, rng)
        return {"energy": np.array([_vqe_exact(n, h, p) for (n, h), p in zip(insts, params)])}
    if kind == "train":
        return None  # the order of the rows is the engine's own shuffle
    dims, w = _network(case, rng)
    a = _round_bf16(torch.from_numpy(_features(case["rows"], case["inputs"], rng)))
    w, off = torch.from_numpy(w).double(), 0
    for k, (i, o) in enumerate(zip(dims[:-1], dims[1:])):
        a = a @ _round_bf16(w[off:off + i * o].view(i, o)) + w[off + i * o:off + i * o + o]
        off += i * o + o
        if k + 2 < len(dims):
            a = _round_bf16(torch.relu(a))
    return {"y": a[:, 0].numpy()}
