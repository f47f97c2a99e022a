"""Density-matrix circuits as programs over the row and column bits, against the gate-by-gate
path (set_circuit_fusion(False)) and, for the compiled gates themselves, against numpy: unitary
and non-unitary gates up to four qubits with controls, depolarizing on one and two qubits, the
channels that stay superoperators, and gates that split a run.  Observables of many terms in
one call against term by term.

Tolerance: either path rounds every entry a few times per gate; a CNOT as H CZ H adds up to
four entries of the result's size, a channel's matrix product up to 16: relative Frobenius
error <= 32 * (gates + 1) * 2^-53."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import qulacs_amd as q
from qulacs_amd import _lib
from qulacs_amd.gate import (
    CNOT, CZ, RX, RZ, SWAP, TOFFOLI, AmplitudeDampingNoise, BitFlipNoise, DenseMatrix, DephasingNoise,
    DepolarizingNoise, DiagonalMatrix, H, IndependentXZNoise, Identity, PauliRotation, Probabilistic, S, T,
    TwoQubitDepolarizingNoise, X, sqrtY, to_matrix_gate)
from tests.golden.gen import haar_unitary
from tests.gpu_util import DevState, cmat

pytestmark = pytest.mark.gpu


def _circuit(rng, n, count, style):
    c = q.QuantumCircuit(n)
    kinds = {"depol": ["u", "h", "rz", "cnot", "cz", "d1", "d2", "d1"],
             "pairs": ["prob2", "prob2", "prob2", "u", "d2", "ad"],  # runs of channels on one pair
             "noise": ["u", "cnot", "d1", "ad", "deph", "bf", "xz", "rx"],
             "all": ["u", "h", "s", "t", "x", "sy", "rz", "cnot", "cz", "swap", "d1", "d2", "ad", "deph", "bf", "xz", "u2", "diag2",
                     "cu", "toffoli", "p0", "prob2", "rot", "id", "u3", "wide"]}[style]
    for _ in range(count):
        kind = kinds[int(rng.integers(len(kinds)))]
        t = [int(x) for x in rng.permutation(n)]
        a, p = float(rng.uniform(0, 6.0)), float(rng.uniform(0, 0.4))
        one = {"h": H, "s": S, "t": T, "x": X, "sy": sqrtY, "id": Identity}
        if kind in one:
            c.add_gate(one[kind](t[0]))
        elif kind in ("d1", "ad", "deph", "bf", "xz"):
            f = {"d1": DepolarizingNoise, "ad": AmplitudeDampingNoise, "deph": DephasingNoise, "bf": BitFlipNoise,
                 "xz": IndependentXZNoise}[kind]
            c.add_gate(f(t[0], p))
        elif kind == "u":
            c.add_gate(DenseMatrix(t[0], haar_unitary(rng, 1)))
        elif kind == "p0":
            c.add_gate(DenseMatrix(t[0], [[1, 0.1], [0.05j, 0.8]]))
        elif kind in ("rx", "rz"):
            c.add_gate((RX if kind == "rx" else RZ)(t[0], a))
        elif n >= 2 and kind in ("cnot", "cz", "swap"):
            c.add_gate({"cnot": CNOT, "cz": CZ, "swap": SWAP}[kind](t[0], t[1]))
        elif n >= 2 and kind == "d2":
            c.add_gate(TwoQubitDepolarizingNoise(t[0], t[1], p))
        elif n >= 2 and kind == "u2":
            c.add_gate(DenseMatrix(t[:2], haar_unitary(rng, 2)))
        elif n >= 2 and kind == "diag2":
            c.add_gate(DiagonalMatrix(t[:2], np.exp(1j * rng.uniform(0, 6, 4)) * [1, 1, 1, 0.9]))
        elif n >= 2 and kind == "cu":
            g = to_matrix_gate(RX(t[0], a))
            g.add_control_qubit(t[1], int(rng.integers(2)))
            c.add_gate(g)
        elif n >= 2 and kind == "prob2":  # leaves a part of the distribution to the identity
            c.add_gate(Probabilistic([p / 2, p / 3], [CNOT(t[0], t[1]), SWAP(t[0], t[1])]))
        elif n >= 3 and kind == "toffoli":
            c.add_gate(TOFFOLI(*t[:3]))
        elif n >= 3 and kind == "u3":
            c.add_gate(DenseMatrix(t[:3], haar_unitary(rng, 3)))
        elif n >= 3 and kind == "rot":
            c.add_gate(PauliRotation(t[:3], [1, 2, 3], a))
        elif n >= 5 and kind == "wide":  # splits the run
            c.add_gate(PauliRotation(t[:5], [1, 2, 3, 1, 2], a))
    return c


def _random_rho(rng, n):
    d = 1 << n
    a = rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d))
    a = a @ a.conj().T
    return a / np.trace(a).real


def _run(c, n, rho, fused):
    q.set_circuit_fusion(fused)
    try:
        s = q.DensityMatrix(n)
        s.load(rho)
        c.update_quantum_state(s)
        first = np.array(s.get_matrix())
        s.load(rho)
        c.update_quantum_state(s)  # the plan that is there
        return first, np.array(s.get_matrix()), s
    finally:
        q.set_circuit_fusion(True)


@pytest.mark.parametrize("n,count,style", [(2, 30, "pairs"), (3, 60, "pairs"), (1, 12, "all"), (2, 7, "depol"), (2, 40, "depol"), (2, 40, "all"), (3, 60, "all"), (4, 80, "noise"),
                                           (5, 120, "depol"), (5, 120, "all"), (6, 150, "noise"), (6, 150, "all"), (7, 200, "depol"),
                                           (7, 160, "all"), (8, 120, "depol"), (11, 30, "all")])
def test_noisy_circuit(n, count, style):
    rng = np.random.default_rng(100 * n + count)
    c = _circuit(rng, n, count, style)
    rho = _random_rho(rng, n)
    want = _run(c, n, rho, False)[0]
    tol = 32 * (count + 1) * 2.0 ** -53 * np.linalg.norm(want)
    for got in _run(c, n, rho, True)[:2]:
        assert np.linalg.norm(got - want) <= tol


def test_parameter_and_state_vector_plans():
    """One circuit on a density matrix and a state vector in turn, with angles changed between."""
    n = 5
    c = q.ParametricQuantumCircuit(n)
    for k in range(n):
        c.add_parametric_RX_gate(k, 0.1 * k)
        c.add_H_gate(k)
    for k in range(n - 1):
        c.add_CNOT_gate(k, k + 1)
    rng = np.random.default_rng(3)
    for _ in range(3):
        for k in range(n):
            c.set_parameter(k, float(rng.uniform(0, 6)))
        sv, dm = q.QuantumState(n), q.DensityMatrix(n)
        c.update_quantum_state(dm)
        c.update_quantum_state(sv)
        psi = np.array(sv.get_vector())
        assert np.linalg.norm(np.array(dm.get_matrix()) - np.outer(psi, psi.conj())) <= 32 * 16 * 2.0 ** -53


@pytest.mark.parametrize("n,bits", [(4, [1, 3]), (6, [0, 3]), (6, [4, 1, 5, 2]), (14, [0, 7, 6, 13]), (14, [7, 0]), (16, [12, 4, 15, 7])])
def test_depolarizing_gate(n, bits):
    rng = np.random.default_rng(n + len(bits))
    psi = rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)
    s, t = 0.7, 0.11
    x = np.arange(1 << n)
    b = [(x >> k) & 1 for k in bits]
    agree = np.logical_and.reduce([b[i] == b[i + 1] for i in range(0, len(bits), 2)])
    mask = sum(1 << k for k in bits)
    total = np.zeros(1 << n, dtype=complex)
    for v in range(1 << (len(bits) // 2)):
        at = sum(((v >> i) & 1) * ((1 << bits[2 * i]) | (1 << bits[2 * i + 1])) for i in range(len(bits) // 2))
        total += psi[(x & ~mask) | at]
    want = s * psi + t * np.where(agree, total, 0)
    g = (_lib.QmBatchGate * 1)()
    g[0].kind, g[0].qubit_count, m = _lib.BATCH_DEPOL, len(bits), cmat([s + 1j * t])
    for i, k in enumerate(bits):
        g[0].qubits[i] = k
    g[0].matrix = C.cast(m, _lib.PC)
    with pytest.raises(_lib.QulacsMI355Error):  # needs blocks of 4
        _lib.call("qm_circuit_create", n, g, 1, 3, 0)
    prog = _lib.call("qm_circuit_create", n, g, 1, 0, 0)
    with DevState.from_host(psi) as d:
        _lib.call("qm_circuit_apply", prog, d.ptr, 1 << n, None, 0)
        got = d.download()
    _lib.call("qm_circuit_destroy", prog)
    assert np.linalg.norm(got - want) <= 8 * 2.0 ** -53 * np.linalg.norm(want)


@pytest.mark.parametrize("n,terms", [(1, 3), (3, 12), (4, 64), (4, 65), (8, 5), (8, 200), (5, 5000)])
def test_observable_in_one_call(n, terms):
    rng = np.random.default_rng(n * 1000 + terms)
    s = q.DensityMatrix(n)
    rho = _random_rho(rng, n)
    s.load(rho)
    op, want, weight = q.GeneralQuantumOperator(n), 0.0, 0.0
    paulis = [np.eye(2), np.array([[0, 1], [1, 0]]), np.array([[0, -1j], [1j, 0]]), np.diag([1, -1])]
    for _ in range(terms):
        ids = [int(i) for i in rng.integers(0, 4, n)]
        co = complex(rng.standard_normal(), rng.standard_normal())
        op.add_operator(co, " ".join(f"{'IXYZ'[i]} {k}" for k, i in enumerate(ids)))
        m = np.eye(1)
        for i in ids:
            m = np.kron(paulis[i], m)
        want += co * np.sum(m.T * rho)
        weight += abs(co)
    # |Tr(P rho)| <= 1: every product and sum rounds at most once per addend
    assert abs(op.get_expectation_value(s) - want) <= 2.0 ** -53 * weight * (4 * np.log2(terms << n) + 8)
