"""The work a user of qulacs_amd has it do, as cases that can be timed and compared.

Eight families, each through the package's public entry points:

* circuit   QuantumCircuit on a fresh state, then an observable and samples (one shot of a
            variational energy, a QAOA run, a random-circuit benchmark);
* gates     gate objects applied one by one to a resident state (interactive use, circuits
            that a program builds and applies gate by gate);
* dm        a noisy circuit on a density matrix;
* batch     many small circuits with their energies in one call (data sets, sweeps);
* adjoint   energies and gradients of a batch of parameter sets through torch.autograd;
* backprop  one step of a variational loop on ParametricQuantumCircuit: new angles, the
            energy and the gradient;
* serving   requests of mixed size through the request server;
* readout   expectation values, probabilities, entropy and samples of a prepared state.

Sizes run from a few qubits, where launches and latency count, to states of several GiB.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import qulacs_amd as q
from qulacs_amd import gate
from qulacs_amd.adjoint import AdjointCircuit, expectation
from qulacs_amd.batch import Batch, pauli_masks
from qulacs_amd.serving import Server

_P = [np.eye(2), np.array([[0, 1], [1, 0]]), np.array([[0, -1j], [1j, 0]]), np.diag([1, -1])]
_P = [np.asarray(p, dtype=np.complex128) for p in _P]


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # one energy of a small variational circuit: a few microseconds of work, so launches,
        # synchronisation and host calls are what counts
        {"name": "circuit_8q", "kind": "circuit", "style": "ansatz", "n": 8, "layers": 4, "terms": 15, "samples": 0},
        # QAOA on a ring with chords: two-qubit phases between layers of mixers; an odd qubit
        # count that leaves most of the chip idle when a state is cut into large tiles
        {"name": "qaoa_17q", "kind": "circuit", "style": "qaoa", "n": 17, "layers": 4, "terms": 25, "samples": 1000},
        # the 20-qubit brickwork benchmark: circuit, 16-term observable, 1024 samples
        {"name": "brickwork_20q", "kind": "circuit", "style": "brickwork", "n": 20, "layers": 10, "terms": 16,
         "samples": 1024},
        # a large random circuit: 1 GiB of amplitudes, arithmetic in the fused executor
        {"name": "brickwork_26q", "kind": "circuit", "style": "brickwork", "n": 26, "layers": 20, "terms": 4,
         "samples": 0},
        # gate by gate on a 4 GiB state: every gate is a pass over memory (dense on 1 to 5
        # qubits, rotations, controlled, diagonal, permutations, Pauli rotations)
        {"name": "gates_28q", "kind": "gates", "n": 28, "count": 24},
        # a small noisy circuit: some hundred launches on 16 KiB
        {"name": "dm_5q", "kind": "dm", "n": 5, "layers": 3, "noise": "Depolarizing", "p": 0.01},
        # a 12-qubit density matrix (256 MiB) with depolarizing noise after every gate
        {"name": "dm_12q", "kind": "dm", "n": 12, "layers": 3, "noise": "Depolarizing", "p": 0.01},
        # a set of small circuits of 8 to 16 qubits with a transverse-field Ising energy each
        {"name": "batch_512", "kind": "batch", "count": 512, "lo": 8, "hi": 16, "layers": 8},
        # gradients of the 20-qubit, 12-layer hardware-efficient ansatz, forward and backward
        {"name": "adjoint_20q", "kind": "adjoint", "n": 20, "layers": 12, "sets": 16},
        # one step of a variational loop through the drop-in class: new angles every step
        {"name": "backprop_12q", "kind": "backprop", "n": 12, "layers": 3, "field": 1.0},
        # 24 requests of 10 to 22 qubits, submitted together and waited for
        {"name": "serving_24", "kind": "serving", "count": 24, "lo": 10, "hi": 22, "depth": 40, "samples": 1000},
        # reading a prepared 25-qubit state out (512 MiB)
        {"name": "readout_25q", "kind": "readout", "n": 25, "terms": 24, "samples": 10000},
    ]


def _log(rng, lo, hi):
    return float("%.3g" % math.exp(rng.uniform(math.log(lo), math.log(hi))))


def _log_int(rng, lo, hi):
    return int(round(_log(rng, lo, hi)))


def draw(rng):
    """Sizes spread over the families' ranges; qubit counts are the logarithm of a state's size."""
    kind = rng.choice(["circuit", "circuit", "circuit", "gates", "dm", "batch", "adjoint", "backprop", "serving",
                       "readout"])
    if kind == "circuit":
        n = rng.randint(4, 26)
        style = rng.choice(["ansatz", "qaoa", "brickwork", "mixed"])
        most = 40 if n <= 24 else 10 * (28 - n)  # at most brickwork_26q's work
        return {"kind": kind, "style": style, "n": n, "layers": _log_int(rng, 2, most), "terms": rng.randint(1, 40),
                "samples": rng.choice([0, _log_int(rng, 1, 5000)])}
    if kind == "gates":
        return {"kind": kind, "n": rng.randint(3, 27), "count": rng.randint(10, 24)}
    if kind == "dm":
        n = rng.randint(2, 12)
        return {"kind": kind, "n": n, "layers": rng.randint(1, 3),
                "noise": rng.choice(["Depolarizing", "AmplitudeDamping"]), "p": _log(rng, 0.001, 0.1)}
    if kind == "batch":
        lo = rng.randint(3, 12)
        return {"kind": kind, "count": _log_int(rng, 4, 512), "lo": lo, "hi": rng.randint(lo, 16),
                "layers": rng.randint(2, 8)}
    if kind == "adjoint":
        n = rng.randint(4, 20)
        return {"kind": kind, "n": n, "layers": rng.randint(2, 12), "sets": _log_int(rng, 1, 16)}
    if kind == "backprop":
        return {"kind": kind, "n": rng.randint(3, 12), "layers": rng.randint(1, 3), "field": round(rng.uniform(0.5, 1.5), 3)}
    if kind == "serving":
        lo = rng.randint(5, 14)
        return {"kind": kind, "count": rng.randint(4, 24), "lo": lo, "hi": rng.randint(lo, 22),
                "depth": _log_int(rng, 8, 40), "samples": _log_int(rng, 10, 1000)}
    return {"kind": kind, "n": rng.randint(4, 25), "terms": rng.randint(1, 24), "samples": _log_int(rng, 1, 10000)}


# ---------------------------------------------------------------- inputs, made from the seed alone
def _haar(rng, k, count):
    """`count` Haar-random unitaries on k qubits."""
    d = 1 << k
    z = rng.standard_normal((count, d, d)) + 1j * rng.standard_normal((count, d, d))
    u, r = np.linalg.qr(z)
    ph = np.diagonal(r, axis1=1, axis2=2)
    return np.ascontiguousarray(u * (ph / np.abs(ph))[:, None, :])


def _random_terms(rng, n, count):
    """(qubits, Pauli ids, coefficient) of random Pauli strings."""
    out = []
    for _ in range(count):
        p = rng.integers(0, 4, size=n)
        if not p.any():
            p[0] = 3
        t = [i for i in range(n) if p[i]]
        out.append((t, [int(p[i]) for i in t], float(rng.standard_normal())))
    return out


def _chain_terms(rng, n, h=None):
    """A transverse-field Ising chain with field h, or one from U[0.5, 1.5]."""
    h = float(rng.uniform(0.5, 1.5)) if h is None else h
    return [([i, i + 1], [3, 3], 1.0) for i in range(n - 1)] + [([i], [1], h) for i in range(n)]


def _circuit_gates(case, rng):
    """A list of (kind, qubits, value): the circuit as data, for the package and for exact()."""
    n, L, style = case["n"], case["layers"], case["style"]
    g = []
    if style == "brickwork":
        u = _haar(rng, 1, n * L)
        for k in range(L):
            g += [("U", [i], u[k * n + i]) for i in range(n)]
            g += [("CNOT", [i, i + 1], None) for i in range(k % 2, n - 1, 2)]
    elif style == "ansatz":
        for _ in range(L):
            for i in range(n):
                g += [("RY", [i], float(rng.uniform(0, 2 * np.pi))), ("RZ", [i], float(rng.uniform(0, 2 * np.pi)))]
            g += [("CZ", [i, i + 1], None) for i in range(n - 1)]
    elif style == "qaoa":
        edges = _edges(n)
        g += [("H", [i], None) for i in range(n)]
        for _ in range(L):
            a, b = float(rng.uniform(0, np.pi)), float(rng.uniform(0, np.pi))
            g += [("ZZ", e, a * w) for e, w in zip(edges, rng.uniform(0.5, 1.5, len(edges)))]
            g += [("RX", [i], b) for i in range(n)]
    else:  # a program's mixture of named, rotation, controlled and dense gates
        for _ in range(L * n):
            kind = ["H", "T", "RX", "RZ", "U", "U", "CNOT", "CZ", "SWAP", "U2", "TOFFOLI", "ZZ"][int(rng.integers(12))]
            k = {"CNOT": 2, "CZ": 2, "SWAP": 2, "U2": 2, "ZZ": 2, "TOFFOLI": 3}.get(kind, 1)
            t = [int(x) for x in rng.choice(n, k, replace=False)]
            v = None
            if kind in ("RX", "RZ", "ZZ"):
                v = float(rng.uniform(0, 2 * np.pi))
            elif kind in ("U", "U2"):
                v = _haar(rng, k, 1)[0]
            g.append((kind, t, v))
    return g


def _edges(n):
    """A ring, with a chord across it from every third qubit."""
    e = [[i, (i + 1) % n] for i in range(n if n > 2 else 1)]
    if n >= 6:
        e += [[i, i + n // 2] for i in range(0, n // 2, 3)]
    return e


_KINDS = ["U", "U2", "U3", "U4", "U5", "RX", "RY", "RZ", "CNOT", "CZ", "SWAP", "H", "T", "ZZ", "XYZ", "CU", "DIAG2",
          "TOFFOLI"]


def _gate_list(case, rng):
    n, g = case["n"], []
    order = list(rng.permutation(len(_KINDS)))
    for j in range(case["count"]):
        kind = _KINDS[order[j % len(order)]]
        k = {"U": 1, "U2": 2, "U3": 3, "U4": 4, "U5": 5, "CNOT": 2, "CZ": 2, "SWAP": 2, "ZZ": 2, "XYZ": 3, "CU": 2,
             "DIAG2": 2, "TOFFOLI": 3}.get(kind, 1)
        if k > n:
            kind, k = "U", 1
        t = [int(x) for x in rng.choice(n, k, replace=False)]
        v = None
        if kind in ("RX", "RY", "RZ", "ZZ", "XYZ"):
            v = float(rng.uniform(0, 2 * np.pi))
        elif kind in ("U", "U2", "U3", "U4", "U5"):
            v = _haar(rng, k, 1)[0]
        elif kind == "CU":
            v = _haar(rng, 1, 1)[0]
        elif kind == "DIAG2":
            v = np.exp(1j * rng.uniform(0, 2 * np.pi, 4))
        g.append((kind, t, v))
    return g


def _as_gate(kind, t, v):
    """The package's gate object."""
    if kind in ("U", "U2", "U3", "U4", "U5"):
        return gate.DenseMatrix(t if len(t) > 1 else t[0], v)
    if kind in ("RX", "RY", "RZ"):
        return getattr(gate, kind)(t[0], v)
    if kind in ("H", "T"):
        return getattr(gate, kind)(t[0])
    if kind in ("CNOT", "CZ", "SWAP"):
        return getattr(gate, kind)(t[0], t[1])
    if kind == "ZZ":
        return gate.PauliRotation(t, [3, 3], v)
    if kind == "XYZ":
        return gate.PauliRotation(t, [1, 2, 3], v)
    if kind == "DIAG2":
        return gate.DiagonalMatrix(t, v)
    m = gate.to_matrix_gate(gate.X(t[-1])) if kind == "TOFFOLI" else gate.DenseMatrix(t[-1], v)  # TOFFOLI, CU
    for c in t[:-1]:
        m.add_control_qubit(c, 1)
    return m


def _as_matrix(kind, t, v):
    """(targets, matrix) with bit i of the matrix index on targets[i]."""
    if kind in ("U", "U2", "U3", "U4", "U5"):
        return t, v
    if kind in ("RX", "RY", "RZ"):  # exp(+i v P / 2)
        p = _P[{"RX": 1, "RY": 2, "RZ": 3}[kind]]
        return t, math.cos(v / 2) * _P[0] + 1j * math.sin(v / 2) * p
    if kind == "H":
        return t, np.array([[1, 1], [1, -1]], dtype=np.complex128) / math.sqrt(2)
    if kind == "T":
        return t, np.diag([1, np.exp(0.25j * np.pi)])
    if kind in ("ZZ", "XYZ"):
        p = np.eye(1)
        for b in ([3, 3] if kind == "ZZ" else [1, 2, 3]):
            p = np.kron(_P[b], p)
        return t, math.cos(v / 2) * np.eye(len(p)) + 1j * math.sin(v / 2) * p
    if kind == "CZ":
        return t, np.diag([1, 1, 1, -1]).astype(np.complex128)
    if kind == "SWAP":
        return t, np.eye(4, dtype=np.complex128)[[0, 2, 1, 3]]
    if kind == "DIAG2":
        return t, np.diag(v)
    m = np.eye(1 << len(t), dtype=np.complex128)  # CNOT, TOFFOLI, CU: controls first, the target last
    u = v if kind == "CU" else _P[1]
    c = (1 << (len(t) - 1)) - 1
    at = [c, c | 1 << (len(t) - 1)]
    m[np.ix_(at, at)] = u
    return t, m


def _circuit_terms(case, rng):
    if case["style"] == "ansatz":
        terms = _chain_terms(rng, case["n"])
    elif case["style"] == "qaoa":
        terms = [(e, [3, 3], 1.0) for e in _edges(case["n"])]
    else:
        terms = _random_terms(rng, case["n"], case["terms"])
    return terms[:max(1, case["terms"])]


def _observable(n, terms):
    o = q.Observable(n)
    for t, p, c in terms:
        o.add_operator(c, " ".join("%s %d" % ("IXYZ"[b], i) for i, b in zip(t, p)))
    return o


class _Memory:
    """A state's device memory as the array interface describes it."""

    def __init__(self, state, entries):
        self.state = state
        self.__cuda_array_interface__ = {"shape": (entries,), "typestr": "<c16", "data": (state.data_ptr(), False),
                                         "version": 2}


def _view(state, entries):
    return torch.as_tensor(_Memory(state, entries), device="cuda")


def _random_vector(n, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    v = torch.randn(2 << n, dtype=torch.float64, device="cuda", generator=g)
    return torch.view_as_complex((v / v.norm()).view(-1, 2))


def _noisy_gates(case, rng):
    """Brickwork layers with a noise channel after every gate, its strength within a factor of two of case["p"]."""
    n, g, p = case["n"], [], case["p"]
    u = _haar(rng, 1, n * case["layers"])
    for k in range(case["layers"]):
        for i in range(n):
            g.append(("U", [i], u[k * n + i], float(rng.uniform(p / 2, 2 * p))))
        for i in range(k % 2, n - 1, 2):
            g.append(("CNOT", [i, i + 1], None, float(rng.uniform(p / 2, 2 * p))))
    return g


def _small_circuits(case, rng):
    """Per circuit: qubits, angles (layers, qubits, 2) of RY then RZ, each layer ending in a CZ chain, and terms."""
    out = []
    for _ in range(case["count"]):
        n = int(rng.integers(case["lo"], case["hi"] + 1))
        L = int(rng.integers(max(1, case["layers"] // 2), case["layers"] + 1))
        out.append((n, rng.uniform(0, 2 * np.pi, (L, n, 2)), _chain_terms(rng, n)))
    return out


def _rot(kind, a):
    c, s = math.cos(a / 2), math.sin(a / 2)
    return np.array([[c, s], [-s, c]]) if kind == "RY" else np.diag([c + 1j * s, c - 1j * s])


def _masks(terms):
    return [(*pauli_masks(t, p), c) for t, p, c in terms]


def _heisenberg(n):
    return [([i, i + 1], [p, p], 1.0) for i in range(n - 1) for p in (1, 2, 3)]


def _ansatz_ops(n, layers):
    """RY, RZ on every qubit and a CZ chain, `layers` times: (kind, qubits, parameter)."""
    ops, k = [], 0
    for _ in range(layers):
        for i in range(n):
            ops += [("RY", [i], k), ("RZ", [i], k + 1)]
            k += 2
        ops += [("CZ", [i, i + 1], None) for i in range(n - 1)]
    return ops, k


def _requests(case, rng):
    out = []
    for _ in range(case["count"]):
        n = int(round(math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"])))))
        depth = int(rng.integers(max(1, case["depth"] // 2), case["depth"] + 1))
        u = _haar(rng, 1, n * depth)
        g = []
        for k in range(depth):
            g += [("dense", [i], u[k * n + i]) for i in range(n)]
            g += [("CNOT", [i, i + 1], None) for i in range(k % 2, n - 1, 2)]
        out.append((n, g, _random_terms(rng, n, 8), rng.random(case["samples"])))
    return out


class _Service:
    """A server as a program holds it: closed when it is no longer used."""

    def __init__(self):
        self.server = Server(hbm_budget_bytes=64 << 30)

    def __del__(self):
        self.server.close()


# ---------------------------------------------------------------- prepare and run
def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind, n = case["kind"], case.get("n", 0)
    s = {"case": case}
    if kind == "circuit":
        c = q.QuantumCircuit(n)
        for g in _circuit_gates(case, rng):
            c.add_gate(_as_gate(*g))
        state = q.QuantumState(n)
        s.update(circuit=c, observable=_observable(n, _circuit_terms(case, rng)), state=state, view=_view(state, 1 << n),
                 seed=int(rng.integers(1 << 30)))
    elif kind == "gates":
        state = q.QuantumState(n)
        v = _view(state, 1 << n)
        v.copy_(_random_vector(n, seed))
        s.update(gates=[_as_gate(*g) for g in _gate_list(case, rng)], state=state, view=v)
    elif kind == "dm":
        c = q.QuantumCircuit(n)
        for k, t, v, p in _noisy_gates(case, rng):
            if case["noise"] == "Depolarizing":
                c.add_noise_gate(_as_gate(k, t, v), "Depolarizing", p)
            else:
                c.add_gate(_as_gate(k, t, v))
                for i in t:
                    c.add_gate(gate.AmplitudeDampingNoise(i, p))
        state = q.DensityMatrix(n)
        s.update(circuit=c, observable=_observable(n, _chain_terms(rng, n)), state=state, view=_view(state, 1 << 2 * n))
    elif kind == "batch":
        b = Batch()
        for m, a, terms in _small_circuits(case, rng):
            g = []
            for layer in a:
                for i in range(m):
                    g += [("dense", [i], _rot("RY", layer[i, 0])), ("dense", [i], _rot("RZ", layer[i, 1]))]
                g += [("CZ", [i, i + 1], None) for i in range(m - 1)]
            b.add(m, g, _masks(terms))
        b.compile(block_qubits=3)  # the width that autotune picks for such circuits
        s.update(batch=b)
    elif kind == "adjoint":
        ops, count = _ansatz_ops(n, case["layers"])
        g = [("CZ", t, None) if k == "CZ" else ("rot", t, [2 if k == "RY" else 3], p, 1.0) for k, t, p in ops]
        theta = torch.from_numpy(rng.uniform(0, 2 * np.pi, (case["sets"], count))).cuda().requires_grad_(True)
        s.update(circuit=AdjointCircuit(n, g, count), theta=theta, terms=_masks(_heisenberg(n)))
    elif kind == "backprop":
        ops, count = _ansatz_ops(n, case["layers"])
        c = q.ParametricQuantumCircuit(n)
        for k, t, p in ops:
            if k == "CZ":
                c.add_CZ_gate(*t)
            else:
                getattr(c, "add_parametric_%s_gate" % k)(t[0], 0.0)
        s.update(circuit=c, state=q.QuantumState(n), observable=_observable(n, _chain_terms(rng, n, case["field"])),
                 theta=[float(x) for x in rng.uniform(0, 2 * np.pi, count)])
    elif kind == "serving":
        s.update(service=_Service(), requests=[(m, g, _masks(t), u) for m, g, t, u in _requests(case, rng)])
    else:
        state = q.QuantumState(n)
        v = _view(state, 1 << n)
        v.copy_(_random_vector(n, seed))
        s.update(state=state, observable=_observable(n, _random_terms(rng, n, case["terms"])),
                 seed=int(rng.integers(1 << 30)), pattern=[int(x) for x in rng.integers(0, 3, n)])
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "circuit":
        st = s["state"]
        st.set_zero_state()
        s["circuit"].update_quantum_state(st)
        out = {"energy": np.float64(s["observable"].get_expectation_value(st)), "state": s["view"]}
        if case["samples"]:
            out["samples"] = np.asarray(st.sampling(case["samples"], s["seed"]), dtype=np.int64)
        return out
    if kind == "gates":
        for g in s["gates"]:
            g.update_quantum_state(s["state"])
        return {"state": s["view"]}
    if kind == "dm":
        st = s["state"]
        st.set_zero_state()
        s["circuit"].update_quantum_state(st)
        return {"energy": np.float64(s["observable"].get_expectation_value(st)), "state": s["view"]}
    if kind == "batch":
        return {"energies": s["batch"].run()}
    if kind == "adjoint":
        s["theta"].grad = None
        e = expectation(s["circuit"], s["theta"], s["terms"])
        e.sum().backward()
        return {"energies": e.detach(), "gradient": s["theta"].grad}
    if kind == "backprop":
        c, st, o = s["circuit"], s["state"], s["observable"]
        for i, a in enumerate(s["theta"]):
            c.set_parameter(i, a)
        st.set_zero_state()
        c.update_quantum_state(st)
        return {"energy": np.float64(o.get_expectation_value(st)), "gradient": np.asarray(c.backprop(o))}
    if kind == "serving":
        srv = s["service"].server
        ids = [srv.submit(*r) for r in s["requests"]]
        got = [srv.wait(i) for i in ids]
        return {"energies": np.asarray([g[0] for g in got]),
                "samples": np.stack([g[1] for g in got]).astype(np.int64)}
    st, n = s["state"], case["n"]
    return {"values": np.asarray([s["observable"].get_expectation_value(st), st.get_squared_norm(),
                                  st.get_marginal_probability(s["pattern"]), st.get_entropy()]),
            "zero": np.asarray([st.get_zero_probability(i) for i in (0, n // 2, n - 1)]),
            "samples": np.asarray(st.sampling(case["samples"], s["seed"]), dtype=np.int64)}


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    """Bytes: the state written (and read) once, results aside.  Flops: 14 per amplitude for a
    2 x 2 matrix on every qubit and layer (4 complex products and 2 sums for a pair), 6 for a
    phase, 8 * 2^k for a dense matrix on k qubits; 4 per amplitude and Pauli term."""
    kind, n = case["kind"], case.get("n", 0)
    N = float(1 << n)
    if kind == "circuit":
        per = {"ansatz": 14.0, "qaoa": 14.0 + 6.0, "brickwork": 14.0, "mixed": 14.0}[case["style"]]
        return {"bytes": 16 * N, "flops": N * (per * n * case["layers"] + 4 * case["terms"])}
    if kind == "gates":
        # each gate is a call of its own and reads and writes what it changes: half of the
        # amplitudes for CNOT, SWAP, T and CU, a quarter for CZ and TOFFOLI: 14.5 of 18 kinds
        return {"bytes": 32 * N * case["count"] * 14.5 / 18, "flops": N * case["count"] * 36.0}
    if kind == "dm":
        return {"bytes": 16 * N * N, "flops": 28 * N * N * n * case["layers"] * 1.5}
    if kind == "batch":
        mean = sum(2.0 ** m * m for m in range(case["lo"], case["hi"] + 1)) / (case["hi"] - case["lo"] + 1)
        return {"bytes": 8.0 * case["count"] * case["layers"] * (case["lo"] + case["hi"]),
                "flops": case["count"] * mean * (14.0 * 0.75 * case["layers"] + 8.0)}
    if kind == "adjoint":
        # forward one 2 x 2 per qubit and layer; backward the same on two states, and two
        # inner products of a Pauli per qubit and layer
        return {"bytes": 32 * N * case["sets"],
                "flops": case["sets"] * N * n * case["layers"] * (14.0 * 3 + 2 * 4.0)}
    if kind == "backprop":
        return {"bytes": 32 * N, "flops": N * n * case["layers"] * (14.0 * 3 + 2 * 4.0)}
    if kind == "serving":
        mean = sum(2.0 ** m * m / m for m in range(case["lo"], case["hi"] + 1)) / sum(
            1.0 / m for m in range(case["lo"], case["hi"] + 1))
        return {"bytes": 16.0 * case["count"] * mean / case["hi"],
                "flops": case["count"] * mean * 14.0 * 0.75 * case["depth"]}
    return {"bytes": 16 * N * 3, "flops": N * (4.0 * case["terms"] + 30.0)}


# Relative error of another complex128 evaluation, from what this path differs from exact() by:
# a state by 6e-16 to 1e-15, and by 1.8e-16 for each CNOT in a fused circuit (3.3e-14 for the 250 of
# brickwork_26q); gradients and vectors of energies by 3e-16 to 5e-16.  The energy of a random
# state is a sum that cancels (2.4e-14 and 5.8e-14 seen with 16 and 4 terms), so the cases that return one
# allow for more terms cancelling.  A uniform within rounding of a step of the cumulative
# distribution may give the neighbouring index.
def tolerance(case):
    t = {"rel": {"circuit": 1e-12, "serving": 4e-13, "dm": 1e-13, "backprop": 1e-13, "readout": 4e-14}.get(case["kind"], 1e-14)}
    if case["kind"] in ("circuit", "serving", "readout"):
        t["differ"] = 0.002
    return t


# ---------------------------------------------------------------- the same in plain torch, 64 bits
def _apply(psi, n, t, m):
    """m (2^k x 2^k, bit i on t[i]) on the last axis of psi, shape (batch, 2^n)."""
    k = len(t)
    if np.count_nonzero(m - np.diag(np.diagonal(m))) == 0 and k == 1:
        v = psi.view(psi.shape[0], -1, 2, 1 << t[0])
        v[:, :, 0] *= complex(m[0, 0])
        v[:, :, 1] *= complex(m[1, 1])
        return psi
    if k == 1:
        v = psi.view(psi.shape[0], -1, 2, 1 << t[0])
        a, b = v[:, :, 0], v[:, :, 1]
        x = complex(m[0, 0]) * a + complex(m[0, 1]) * b
        b.mul_(complex(m[1, 1])).add_(a, alpha=complex(m[1, 0]))
        a.copy_(x)
        return psi
    o = sorted(range(k), key=lambda i: t[i])  # matrix bits in the order of ascending qubits
    idx = np.zeros(1 << k, dtype=np.int64)
    for j in range(1 << k):
        idx[j] = sum(((j >> r) & 1) << o[r] for r in range(k))
    m = m[np.ix_(idx, idx)]
    st = [t[i] for i in o]
    shape, hi = [psi.shape[0]], n
    for x in reversed(st):
        shape += [1 << (hi - x - 1), 2]
        hi = x
    shape.append(1 << hi)
    v = psi.view(shape)
    axes = [2 + 2 * r for r in range(k)]  # most significant first
    front = v.movedim(axes, list(range(k))).contiguous()
    w = torch.matmul(torch.from_numpy(np.ascontiguousarray(m)).to(psi.device), front.view(1 << k, -1)).view(front.shape)
    v.copy_(w.movedim(list(range(k)), axes))
    return psi


def _zero(n):
    psi = torch.zeros(1, 1 << n, dtype=torch.complex128, device="cuda")
    psi[0, 0] = 1
    return psi


def _pauli(psi, n, t, p):
    """P psi for a Pauli string."""
    out = psi.clone()
    for i, b in zip(t, p):
        v = out.view(out.shape[0], -1, 2, 1 << i)
        if b == 3:
            v[:, :, 1] *= -1
            continue
        v = v.flip(2)
        if b == 2:
            v[:, :, 0] *= -1j
            v[:, :, 1] *= 1j
        out = v.reshape(psi.shape)
    return out


def _energy(psi, n, terms):
    return sum(c * (psi.conj() * _pauli(psi, n, t, p)).sum(1).real for t, p, c in terms)


def _phases(n):
    """The signs of a CZ chain."""
    i = torch.arange(1 << n, device="cuda")
    b = i & (i >> 1)
    for s in (16, 8, 4, 2, 1):
        b = b ^ (b >> s)
    return 1.0 - 2.0 * (b & 1).double()


def _adjoint_exact(n, layers, theta, terms):
    """Energies and gradients of the ansatz for theta (sets, parameters), gate by gate."""
    sign = _phases(n)
    sets = theta.shape[0]

    def rot(psi, i, kind, a):
        c, s = torch.cos(a / 2)[:, None, None], torch.sin(a / 2)[:, None, None]
        v = psi.view(sets, -1, 2, 1 << i)
        x, y = v[:, :, 0], v[:, :, 1]
        if kind == "RY":
            w = c * x + s * y
            y.copy_(c * y - s * x)
            x.copy_(w)
        else:
            x.mul_(c + 1j * s)
            y.mul_(c - 1j * s)

    psi = torch.zeros(sets, 1 << n, dtype=torch.complex128, device="cuda")
    psi[:, 0] = 1
    for k in range(layers):
        for i in range(n):
            rot(psi, i, "RY", theta[:, (k * n + i) * 2])
            rot(psi, i, "RZ", theta[:, (k * n + i) * 2 + 1])
        psi *= sign
    lam = torch.zeros_like(psi)
    for t, p, c in terms:
        lam += c * _pauli(psi, n, t, p)
    e = (psi.conj() * lam).sum(1).real
    grad = torch.zeros_like(theta)
    for k in reversed(range(layers)):
        psi *= sign
        lam *= sign
        for i in reversed(range(n)):
            for j, kind, b in ((1, "RZ", 3), (0, "RY", 2)):
                at = (k * n + i) * 2 + j
                grad[:, at] = -(lam.conj() * _pauli(psi, n, [i], [b])).sum(1).imag
                rot(psi, i, kind, -theta[:, at])
                rot(lam, i, kind, -theta[:, at])
    return e, grad


def exact(case, seed):
    rng = np.random.default_rng(seed)
    kind, n = case["kind"], case.get("n", 0)
    if kind == "circuit":
        psi = _zero(n)
        for g in _circuit_gates(case, rng):
            psi = _apply(psi, n, *_as_matrix(*g))
        out = {"energy": np.float64(_energy(psi, n, _circuit_terms(case, rng)).item()), "state": psi[0]}
        if case["samples"]:
            out["samples"] = None
        return out
    if kind == "gates":
        psi = _random_vector(n, seed).view(1, -1)
        for g in _gate_list(case, rng):
            psi = _apply(psi, n, *_as_matrix(*g))
        return {"state": psi[0]}
    if kind == "dm":
        rho = _zero(2 * n)  # row bits above column bits

        def channel(t, kraus):
            s = sum(np.kron(k, k.conj()) for k in kraus)
            return _apply(rho, 2 * n, t + [x + n for x in t], s)

        for k, t, v, p in _noisy_gates(case, rng):
            m = _as_matrix(k, t, v)[1]
            rho = channel(t, [m])
            if case["noise"] == "Depolarizing":
                ops = _P if len(t) == 1 else [np.kron(b, a) for b in _P for a in _P]
                w = [1 - p] + [p / (len(ops) - 1)] * (len(ops) - 1)
                rho = channel(t, [math.sqrt(x) * o for x, o in zip(w, ops)])
            else:
                for i in t:
                    rho = channel([i], [np.diag([1, math.sqrt(1 - p)]).astype(np.complex128),
                                        np.array([[0, math.sqrt(p)], [0, 0]], dtype=np.complex128)])
        e = 0.0
        for t, p, c in _chain_terms(rng, n):  # P acts on the row bits
            e += c * _pauli(rho, 2 * n, [x + n for x in t], p).view(1 << n, 1 << n).diagonal().sum().real.item()
        return {"energy": np.float64(e), "state": rho[0]}
    if kind == "batch":
        found, signs = [], {}
        for m, a, terms in _small_circuits(case, rng):
            sign = signs.setdefault(m, _phases(m))
            psi = _zero(m)
            for layer in a:
                for i in range(m):
                    psi = _apply(psi, m, [i], _rot("RZ", layer[i, 1]) @ _rot("RY", layer[i, 0]))
                psi = psi * sign
            # Z Z terms from the probabilities, X terms from pairs
            prob = (psi[0].abs() ** 2).view(-1)
            e = 0.0
            for t, p, c in terms:
                if p[0] == 3:
                    v = prob.view(-1, 2, 2, 1 << t[0]).sum((0, 3))
                    e = e + c * (v[0, 0] + v[1, 1] - v[0, 1] - v[1, 0])
                else:
                    v = psi.view(-1, 2, 1 << t[0])
                    e = e + 2 * c * (v[:, 0].conj() * v[:, 1]).sum().real
            found.append(e)
        return {"energies": torch.stack(found)}
    if kind == "adjoint":
        theta = torch.from_numpy(rng.uniform(0, 2 * np.pi, (case["sets"], 2 * n * case["layers"]))).cuda()
        e, g = _adjoint_exact(n, case["layers"], theta, _heisenberg(n))
        return {"energies": e, "gradient": g}
    if kind == "backprop":
        terms = _chain_terms(rng, n, case["field"])
        theta = torch.from_numpy(rng.uniform(0, 2 * np.pi, 2 * n * case["layers"])).cuda().view(1, -1)
        e, g = _adjoint_exact(n, case["layers"], theta, terms)
        return {"energy": np.float64(e.item()), "gradient": g[0]}
    if kind == "serving":
        found = []
        for m, g, terms, _ in _requests(case, rng):
            psi = _zero(m)
            for k, t, v in g:
                psi = _apply(psi, m, *_as_matrix("U" if k == "dense" else k, t, v))
            found.append(_energy(psi, m, terms))
        return {"energies": torch.cat(found), "samples": None}
    psi = _random_vector(n, seed).view(1, -1)
    terms = _random_terms(rng, n, case["terms"])
    rng.integers(1 << 30)
    pattern = [int(x) for x in rng.integers(0, 3, n)]
    prob = psi[0].real ** 2 + psi[0].imag ** 2
    keep = prob.view([2] * n)
    for i, b in enumerate(pattern):  # axis of qubit i in what is left: the highest first
        if b < 2:
            keep = keep.narrow(n - 1 - i, b, 1)
    return {"values": torch.stack([_energy(psi, n, terms)[0], prob.sum(), keep.sum(), -(prob * torch.log(prob)).sum()]),
            "zero": torch.stack([prob.view(-1, 2, 1 << i)[:, 0].sum() for i in (0, n // 2, n - 1)]),
            "samples": None}
