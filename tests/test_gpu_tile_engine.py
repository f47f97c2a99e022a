"""The tile engine at the edges of its windows (12 and 13 qubits) and of its
operation encodings: diagonal gates and CZ to qubits outside the window, Z
rotations, shears, CNOT ladders, dense gates of every width; the fused executor
and the batched executor against a gate-by-gate evolution in numpy complex128.

Tolerance: both sides round every gate once per amplitude, and a fused matrix rounds
its entries once per gate: relative 2-norm error <= 4 * (gates + 1) * 2^-53."""
from __future__ import annotations

import numpy as np
import pytest

from qulacs_amd.batch import Batch, FusedCircuit, pauli_masks
from tests.golden.gen import haar_unitary
from tests.gpu_util import DevState

pytestmark = pytest.mark.gpu


def _apply(psi, n, kind, q, m):
    if kind == "CZ":
        kind, m = "diag", np.array([1, 1, 1, -1], dtype=complex)
    elif kind == "CNOT":
        kind, m = "dense", np.eye(4, dtype=complex)[[0, 3, 2, 1]]
    x = np.arange(psi.size)
    row = sum(((x >> t) & 1) << i for i, t in enumerate(q))
    if kind == "diag":
        return psi * np.asarray(m)[row]
    mask = sum(1 << t for t in q)
    m = np.asarray(m).reshape(1 << len(q), -1)
    out = np.zeros_like(psi)
    for c in range(m.shape[0]):
        out += m[row, c] * psi[(x & ~mask) | sum(((c >> i) & 1) << t for i, t in enumerate(q))]
    return out


def _gates(rng, n, count, style, widest):
    g = []
    for _ in range(count):
        kind = {"chain": ["u", "u", "cz1", "cnot1"], "phases": ["u", "zz", "rz", "cz", "diag2", "zzz", "cphase"],
                "all": ["u", "u", "x", "p0", "rz", "cz", "cnot", "zz", "diag2", "diag3", "diag4", "u2", "uk", "swap"]}[style]
        kind = kind[int(rng.integers(len(kind)))]
        pick = lambda k: [int(t) for t in rng.choice(n, k, replace=False)]  # noqa: E731
        a = float(rng.uniform(0, 2 * np.pi))
        if kind == "u":
            g.append(("dense", pick(1), haar_unitary(rng, 1)))
        elif kind == "x":
            g.append(("dense", pick(1), np.array([[0, 1], [1, 0]])))
        elif kind == "p0":  # not unitary: projects a little
            g.append(("dense", pick(1), np.array([[1, 0.1], [0, 0.9]])))
        elif kind == "rz":
            g.append(("diag", pick(1), np.exp([0.5j * a, -0.5j * a])))
        elif kind in ("cz1", "cnot1"):
            t = int(rng.integers(n - 1))
            g.append(("CZ" if kind == "cz1" else "CNOT", [t, t + 1], None))
        elif kind in ("cz", "cnot"):
            g.append((kind.upper(), pick(2), None))
        elif kind in ("zz", "zzz"):
            k = min(n, len(kind))
            par = np.array([bin(i).count("1") & 1 for i in range(1 << k)])
            g.append(("diag", pick(k), np.exp(0.5j * a * (1 - 2 * par))))
        elif kind == "cphase":
            g.append(("diag", pick(2), np.array([1, 1, 1, np.exp(1j * a)])))
        elif kind.startswith("diag"):
            k = int(kind[4])
            d = np.exp(1j * rng.uniform(0, 2 * np.pi, 1 << k))
            g.append(("diag", pick(k), d * (rng.uniform(0.9, 1.1, 1 << k) if rng.random() < 0.3 else 1)))
        elif kind == "swap":
            g.append(("dense", pick(2), np.eye(4)[[0, 2, 1, 3]]))
        else:
            k = 2 if kind == "u2" else int(rng.integers(2, widest + 1))
            g.append(("dense", pick(k), haar_unitary(rng, k)))
    return g


def _random_state(rng, n):
    v = rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)
    return v / np.linalg.norm(v)


@pytest.mark.parametrize("n,count,style,block,window", [
    (4, 40, "all", 0, 0), (9, 80, "phases", 3, 8), (12, 60, "all", 0, 0), (13, 150, "chain", 0, 0), (13, 60, "all", 4, 13),
    (13, 60, "phases", 2, 9), (14, 120, "phases", 0, 0), (15, 80, "all", 4, 12), (16, 200, "chain", 3, 12),
    (17, 90, "phases", 3, 13), (17, 60, "all", 2, 12), (20, 60, "all", 0, 0), (20, 20, "chain", 0, 0)])
def test_fused_circuit(n, count, style, block, window):
    rng = np.random.default_rng(1000 * n + count)
    gates = _gates(rng, n, count, style, block or 3)
    psi = _random_state(rng, n)
    fc = FusedCircuit(n, gates, block, window)
    with DevState.from_host(psi) as s:
        fc.apply(s.ptr)
        got = s.download()
    fc.close()
    for g in gates:
        psi = _apply(psi, n, *g)
    err = np.linalg.norm(got - psi) / np.linalg.norm(psi)
    print(n, style, fc.n, err, flush=True)
    assert err <= 4 * (count + 1) * 2.0 ** -53


@pytest.mark.parametrize("k", [2, 3])
@pytest.mark.parametrize("moduli", ["common", "per qubit", "any"])
def test_diagonal_moduli_near_one(moduli, k):
    """Diagonal entries a few ten units of the last place off the unit circle are applied as given:
    20 gates of modulus 1 + 9e-15 are 1.8e-13 away from 20 phases."""
    rng = np.random.default_rng(5 * k + len(moduli))
    n = 13
    gates = [("dense", [t], haar_unitary(rng, 1)) for t in range(0, n, 2)]
    for i in range(20):
        q = [int(t) for t in rng.choice(n, k, replace=False)]
        bits = (np.arange(1 << k)[:, None] >> np.arange(k)) & 1
        r = {"common": 9e-15 + 0 * bits[:, 0], "per qubit": 4e-15 + 4e-15 * bits[:, 0],
             "any": rng.uniform(0, 9e-15, 1 << k)}[moduli]
        # phases of one Z string beside those of single qubits, so that the gate may become a ZROT
        phase = bits @ rng.uniform(0, 2, k) + (1 - 2 * (bits[:, 0] ^ bits[:, 1])) * rng.uniform(0, 2)
        gates.append(("diag", q, (1 + r) * np.exp(1j * phase)))
    psi = _random_state(rng, n)
    fc = FusedCircuit(n, gates)
    with DevState.from_host(psi) as s:
        fc.apply(s.ptr)
        got = s.download()
    fc.close()
    for g in gates:
        psi = _apply(psi, n, *g)
    err = np.linalg.norm(got - psi) / np.linalg.norm(psi)
    print(moduli, k, err, flush=True)
    assert err <= 4 * (len(gates) + 1) * 2.0 ** -53


@pytest.mark.parametrize("style", ["chain", "phases", "all"])
def test_batch_of_uneven_circuits(style):
    """Sizes on both sides of one tile together; each circuit's energy and state, and the
    energy alone in a batch bit for bit."""
    rng = np.random.default_rng(77)
    sizes = [3, 4, 8, 11, 12, 13, 14, 16]
    work = []
    for n in sizes:
        gates = _gates(rng, n, 6 * n, style if n > 3 else "chain", 3)
        terms = [(*pauli_masks(range(n), rng.integers(0, 4, n)), float(rng.standard_normal())) for _ in range(5)]
        work.append((n, gates, terms))
    b = Batch()
    for n, gates, terms in work:
        b.add(n, gates, terms)
    b.compile(3, keep_states=True)
    e = b.run()
    assert np.array_equal(b.run(), e)
    for i, (n, gates, terms) in enumerate(work):
        psi = np.zeros(1 << n, dtype=complex)
        psi[0] = 1
        for g in gates:
            psi = _apply(psi, n, *g)
        tol = 4 * (len(gates) + 1) * 2.0 ** -53
        assert np.linalg.norm(b.state(i) - psi) <= tol * np.linalg.norm(psi), n
        x = np.arange(1 << n)
        want = 0.0
        for bf, pf, rot, c in terms:
            y = x ^ bf
            sign = 1 - 2 * np.array([bin(int(v) & pf).count("1") & 1 for v in y])
            want += c * np.vdot(psi, (1j ** rot) * sign * psi[y]).real
        assert abs(e[i] - want) <= 2 * tol * sum(abs(t[3]) for t in terms), n
        alone = Batch()
        alone.add(n, gates, terms)
        alone.compile(3)
        assert alone.run()[0] == e[i], n
        alone.close()
    b.close()
