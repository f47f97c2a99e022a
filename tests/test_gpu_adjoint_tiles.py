"""qm_adjoint_* at the edges of its tiles (windows of 11 and 12 qubits, states
below 4 qubits, several parameter sets, more operations than one stage takes)
against a gate-by-gate adjoint in numpy complex128.

Tolerance: both sides round every gate, so amplitudes differ by at most about
gates * 2^-53 * sqrt(2); energies and gradients are sums over the observable's
coefficients: |d| <= 4 * gates * 2^-53 * sum|c| * max|coef|."""
from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from qulacs_amd.adjoint import AdjointCircuit  # noqa: E402
from qulacs_amd.batch import pauli_masks  # noqa: E402
from tests.golden.gen import haar_unitary  # noqa: E402

pytestmark = pytest.mark.gpu


def _pauli(psi, bf, pf, rot):
    """i^rot X^bf Z^pf |psi>, the mask form of a Pauli string."""
    y = np.arange(psi.size, dtype=np.uint64) ^ np.uint64(bf)
    par = np.zeros(psi.size, dtype=np.int64)
    for q in range(int(psi.size).bit_length()):
        if (pf >> q) & 1:
            par ^= ((y >> np.uint64(q)) & np.uint64(1)).astype(np.int64)
    return (1j ** rot) * (1 - 2 * par) * psi[y.astype(np.int64)]


def _matrix(g):
    k = len(g[1])
    if g[0] == "CZ":
        return np.diag([1, 1, 1, -1]).astype(complex)
    if g[0] == "CNOT":
        return np.eye(4, dtype=complex)[[0, 3, 2, 1]]
    return np.diag(g[2]) if g[0] == "diag" else np.asarray(g[2]).reshape(1 << k, 1 << k)


def _dense(psi, n, targets, m):
    out = np.zeros_like(psi)
    x = np.arange(psi.size)
    row = sum(((x >> t) & 1) << i for i, t in enumerate(targets))
    mask = sum(1 << t for t in targets)
    for c in range(m.shape[0]):
        src = (x & ~mask) | sum(((c >> i) & 1) << t for i, t in enumerate(targets))
        out += m[row, c] * psi[src]
    return out


def _reference(n, gates, theta, terms, dtype=complex):
    masks = {i: pauli_masks(g[1], g[2]) for i, g in enumerate(gates) if g[0] == "rot"}

    def rot(psi, i, sign):
        a = sign * gates[i][4] * theta[gates[i][3]] / 2
        return np.cos(a) * psi + 1j * np.sin(a) * _pauli(psi, *masks[i])

    psi = np.zeros(1 << n, dtype=dtype)
    psi[0] = 1
    for i, g in enumerate(gates):
        psi = rot(psi, i, 1) if g[0] == "rot" else _dense(psi, n, g[1], _matrix(g))
    lam = sum((c * _pauli(psi, bf, pf, r) for bf, pf, r, c in terms), np.zeros_like(psi))
    e = np.vdot(psi, lam).real
    grad = np.zeros(len(theta), dtype=theta.dtype)
    for i in reversed(range(len(gates))):
        g = gates[i]
        if g[0] == "rot":
            grad[g[3]] -= g[4] * np.vdot(lam, _pauli(psi, *masks[i])).imag
            psi, lam = rot(psi, i, -1), rot(lam, i, -1)
        else:
            m = _matrix(g).conj().T
            psi, lam = _dense(psi, n, g[1], m), _dense(lam, n, g[1], m)
    return e, grad


def _random_gates(rng, n, count, params):
    gates = []
    for _ in range(count):
        kind = ["rot", "rot", "rot", "dense", "diag", "CZ", "CNOT", "dense2", "diag2"][int(rng.integers(9))]
        if kind == "rot":
            k = int(rng.integers(1, min(n, 4) + 1))
            q = [int(x) for x in rng.choice(n, k, replace=False)]
            gates.append(("rot", q, [int(x) for x in rng.integers(1, 4, k)], int(rng.integers(params)),
                          float(rng.uniform(-2, 2))))
        elif kind in ("dense", "diag") or n == 1:
            m = haar_unitary(rng, 1) if kind == "dense" else np.exp(1j * rng.uniform(0, 6, 2))
            gates.append(("dense" if kind == "dense" else "diag", [int(rng.integers(n))], m))
        else:
            q = [int(x) for x in rng.choice(n, 2, replace=False)]
            m = haar_unitary(rng, 2) if kind == "dense2" else np.exp(1j * rng.uniform(0, 6, 4)) if kind == "diag2" else None
            gates.append(({"dense2": "dense", "diag2": "diag"}.get(kind, kind), q, m))
    return gates


@pytest.mark.parametrize("n,count,sets", [(1, 12, 3), (2, 20, 1), (3, 30, 2), (4, 30, 5), (7, 60, 2), (10, 120, 1),
                                          (11, 240, 2), (12, 100, 1), (13, 150, 2), (15, 80, 3)])
def test_adjoint_matches_gate_by_gate(n, count, sets):
    rng = np.random.default_rng(100 * n + count)
    params = 9
    gates = _random_gates(rng, n, count, params)
    terms = []
    for _ in range(7):
        p = rng.integers(0, 4, n)
        terms.append((*pauli_masks(range(n), p), float(rng.standard_normal())))
    theta = rng.uniform(0, 2 * np.pi, (sets, params))
    e, g = AdjointCircuit(n, gates, params).run(torch.tensor(theta, device="cuda:0"), terms)
    e, g = e.cpu().numpy(), g.cpu().numpy()
    tol = 4 * count * 2.0 ** -53 * sum(abs(t[3]) for t in terms) * 2
    for b in range(sets):
        we, wg = _reference(n, gates, theta[b], terms)
        assert abs(e[b] - we) <= tol, (b, e[b] - we, tol)
        assert np.abs(g[b] - wg).max() <= tol * count / params, (b, np.abs(g[b] - wg).max(), tol)


@pytest.mark.parametrize("n,sets", [(5, 3), (12, 2)])
def test_more_operations_than_the_partial_sums_hold(n, sets):
    """Some 700 operations with gradients (512 share the workspace's columns), the last ones behind
    fixed gates only: gradients as a shorter sweep gives them."""
    rng = np.random.default_rng(n)
    gates = [("dense", [q], haar_unitary(rng, 1)) for q in range(n)]
    params = 40
    while sum(g[0] == "rot" for g in gates) < 700:
        gates += [("rot", [int(rng.integers(n))], [int(rng.integers(1, 4))], int(rng.integers(params)), 1.0),
                  ("CZ", [int(x) for x in rng.choice(n, 2, replace=False)], None)]
    terms = [(3, 3, 2, 1.0), (0, 1 << (n - 1), 0, -0.5)]
    theta = rng.uniform(0, 2 * np.pi, (sets, params))
    circ = AdjointCircuit(n, gates, params)
    e, g = circ.run(torch.tensor(theta, device="cuda:0"), terms)
    e, g = e.cpu().numpy(), g.cpu().numpy()
    tol = 4 * len(gates) * 2.0 ** -53 * 1.5
    for b in range(sets):
        we, wg = _reference(n, gates, theta[b], terms)
        assert abs(e[b] - we) <= tol
        assert np.abs(g[b] - wg).max() <= tol * 700 / params, np.abs(g[b] - wg).max()


def test_non_unitary_fixed_gate_keeps_its_own_operation():
    """A projection between two rotations: its conjugate transpose stands for its
    inverse, as for any fixed gate."""
    n = 4
    gates = [("rot", [0], [2], 0, 1.0), ("dense", [0], np.array([[1, 0.5], [0, 0.25]])), ("rot", [0], [1], 1, 1.0),
             ("CZ", [0, 2], None), ("rot", [2], [2], 2, 1.0)]
    terms = [(1, 0, 0, 1.0), (0, 5, 0, 0.5)]
    theta = np.array([[0.3, 1.1, 2.0]])
    e, g = AdjointCircuit(n, gates, 3).run(torch.tensor(theta, device="cuda:0"), terms)
    we, wg = _reference(n, gates, theta[0], terms)
    assert abs(e.item() - we) < 1e-14 and np.abs(g.cpu().numpy()[0] - wg).max() < 1e-14


@pytest.mark.parametrize("style", ["cnot", "cz", "pauli"])
def test_error_is_that_of_a_gate_by_gate_sweep(style):
    """Gradients against 80 bits: CNOTs, Pauli strings and merged rotations may cost no more than the
    rounding of the same gates one after another in double (rms over 6 circuits, with a fifth for
    chance; Hadamards rounded to double were three times that)."""
    n = 6
    mine, plain = [], []
    for seed in range(6):
        rng = np.random.default_rng(seed)
        gates, params = [], 0
        for _ in range(12):
            for q in range(n):
                for p in (2, 3):
                    gates.append(("rot", [q], [p], params, 1.0))
                    params += 1
            for q in range(n - 1):
                if style == "pauli":
                    gates.append(("rot", [q, q + 1], [int(x) for x in rng.integers(1, 4, 2)], params, 1.0))
                    params += 1
                else:
                    gates.append((style.upper(), [q, q + 1], None))
        terms = []
        for q in range(n - 1):
            m = 3 << q
            terms += [(m, 0, 0, 1.0), (m, m, 2, 1.0), (0, m, 0, 1.0)]
        theta = rng.uniform(0, 2 * np.pi, params)
        _, exact = _reference(n, gates, theta.astype(np.longdouble), terms, np.clongdouble)
        _, double = _reference(n, gates, theta, terms)
        _, g = AdjointCircuit(n, gates, params).run(torch.tensor(theta[None], device="cuda:0"), terms)
        norm = np.linalg.norm(exact.astype(float))
        mine.append(np.linalg.norm((g.cpu().numpy()[0] - exact).astype(float)) / norm)
        plain.append(np.linalg.norm((double - exact).astype(float)) / norm)
    rms = [float(np.sqrt(np.mean(np.square(x)))) for x in (mine, plain)]
    print(style, rms, flush=True)
    assert rms[0] <= 1.2 * rms[1]


def test_result_does_not_depend_on_the_batch():
    n = 9
    rng = np.random.default_rng(5)
    gates = _random_gates(rng, n, 70, 5)
    terms = [(3, 3, 2, 1.0), (0, 1 << 8, 0, -0.5)]
    theta = torch.tensor(rng.uniform(0, 6, (6, 5)), device="cuda:0")
    circ = AdjointCircuit(n, gates, 5)
    e, g = circ.run(theta, terms)
    for b in range(6):
        e1, g1 = circ.run(theta[b:b + 1], terms)
        assert torch.equal(e1[0], e[b]) and torch.equal(g1[0], g[b])
