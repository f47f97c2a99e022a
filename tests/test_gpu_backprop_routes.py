"""ParametricQuantumCircuit.backprop through the adjoint engine and through the gate-by-gate
walk (set_circuit_fusion(False)) on the same circuits: every kind of gate that the engine
takes, gates it does not take (a three-qubit matrix, a controlled rotation), rotations that
are no parameter, edits between calls, and copies.

Tolerance: both walk the same gates in complex128: |d| <= 16 * gates * 2^-53 * sum|c|."""
from __future__ import annotations

import numpy as np
import pytest

import qulacs_amd as q
from qulacs_amd import gate
from tests.golden.gen import haar_unitary

pytestmark = pytest.mark.gpu


def _both(c, obs, scale):
    fused = np.array(c.backprop(obs))
    again = np.array(c.backprop(obs))
    q.set_circuit_fusion(False)
    try:
        walk = np.array(c.backprop(obs))
    finally:
        q.set_circuit_fusion(True)
    assert np.array_equal(fused, again)
    assert fused.shape == walk.shape == (c.get_parameter_count(),)
    assert np.abs(fused - walk).max() <= 16 * c.get_gate_count() * 2.0 ** -53 * scale
    return fused


def _observable(rng, n, terms):
    o = q.Observable(n)
    scale = 0.0
    for _ in range(terms):
        p = rng.integers(0, 4, n)
        c = float(rng.standard_normal())
        scale += abs(c)
        o.add_operator(c, " ".join(f"{'IXYZ'[b]} {i}" for i, b in enumerate(p)))
    return o, scale


@pytest.mark.parametrize("n,extra", [(1, ""), (2, ""), (5, ""), (5, "dense3"), (5, "controlled"), (11, ""), (13, "")])
def test_backprop_routes_agree(n, extra):
    rng = np.random.default_rng(n)
    c = q.ParametricQuantumCircuit(n)
    for i in range(n):
        c.add_parametric_RX_gate(i, float(rng.uniform(0, 6)))
        c.add_H_gate(i)
        c.add_parametric_RY_gate(i, float(rng.uniform(0, 6)))
        c.add_T_gate(i)
        c.add_gate(gate.ParametricRZ(i, 0.4))  # not registered as a parameter
        c.add_dense_matrix_gate([i], haar_unitary(rng, 1))
    if n > 1:
        c.add_CNOT_gate(0, n - 1)
        c.add_SWAP_gate(0, 1)
        c.add_parametric_multi_Pauli_rotation_gate([0, n - 1], [3, 3], 0.3)
        c.add_dense_matrix_gate([n - 1, 0], haar_unitary(rng, 2))
        c.add_CZ_gate(1, 0)
    if n > 3:
        c.add_parametric_multi_Pauli_rotation_gate([0, 1, 2, 3], [1, 2, 3, 1], 1.3)
    if extra == "dense3":
        c.add_dense_matrix_gate([2, 0, 1], haar_unitary(rng, 3))
    if extra == "controlled":
        g = gate.DenseMatrix(0, haar_unitary(rng, 1))
        g.add_control_qubit(1, 0)
        c.add_gate(g)
    c.add_parametric_RZ_gate(0, 0.9)
    c.add_parametric_RX_gate(0, 0.2)
    obs, scale = _observable(rng, n, 6)
    first = _both(c, obs, scale)
    for i in range(c.get_parameter_count()):
        c.set_parameter(i, float(rng.uniform(0, 6)))
    second = _both(c, obs, scale)
    assert np.abs(first - second).max() > 1e-6
    copy = c.copy()
    assert np.array_equal(np.array(copy.backprop(obs)), second)
    c.remove_gate(c.get_gate_count() - 1)
    c.add_X_gate(0)
    _both(c, obs, scale)


def test_backprop_with_a_complex_operator_keeps_the_walk():
    n = 3
    c = q.ParametricQuantumCircuit(n)
    for i in range(n):
        c.add_parametric_RY_gate(i, 0.3 + i)
    o = q.GeneralQuantumOperator(n)
    o.add_operator(1.0 + 0.5j, "X 0")
    o.add_operator(0.25, "Z 1")
    _both(c, o, 2.0)


def _rings(n, count):
    out = []
    for k in range(count):
        c = q.ParametricQuantumCircuit(n)
        for i in range(n):
            c.add_parametric_RX_gate(i, 0.1 + 0.05 * k + 0.01 * i)
            c.add_CNOT_gate(i, (i + 1) % n)
        out.append(c)
    return out


def test_circuits_share_their_workspaces():
    """40 circuits that have run backprop hold their tables (some KiB), not a stream with 16 MiB of
    scratch and a workspace each; the last one to go gives the rest back."""
    torch = pytest.importorskip("torch")
    torch.cuda.init()
    obs = q.Observable(8)
    obs.add_operator(1.0, "Z 0 Z 3")
    for c in _rings(8, 2):  # the runtime's own first allocations
        c.backprop(obs)
    del c
    free = [torch.cuda.mem_get_info()[0]]
    circuits = _rings(8, 40)
    for c in circuits:
        c.backprop(obs)
    free.append(torch.cuda.mem_get_info()[0])
    del circuits, c
    free.append(torch.cuda.mem_get_info()[0])
    print([(free[0] - f) >> 20 for f in free], flush=True)
    # tables: 15 allocations a circuit, which the runtime rounds to at most 64 KiB
    assert free[0] - free[1] < (32 << 20) + 40 * 15 * (64 << 10)
    assert free[0] - free[2] < 8 << 20


def test_threads_with_circuits_of_their_own():
    from concurrent.futures import ThreadPoolExecutor

    rng = np.random.default_rng(8)
    obs, _ = _observable(rng, 9, 5)
    circuits = _rings(9, 6)
    want = [c.backprop(obs) for c in circuits]
    with ThreadPoolExecutor(6) as ex:
        for _ in range(4):
            assert list(ex.map(lambda c: c.backprop(obs), circuits)) == want
