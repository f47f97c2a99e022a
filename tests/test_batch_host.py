"""Host-side validation of the batched-circuit entry points (no device work)."""
from __future__ import annotations

import numpy as np
import pytest

from qulacs_amd._lib import QulacsMI355Error
from qulacs_amd.batch import Batch, pauli_masks


def test_pauli_masks_match_reference_form():
    # X on 0, Y on 2, Z on 3 -> bit flip {0, 2}, phase flip {2, 3}, one Y
    assert pauli_masks([0, 2, 3], [1, 2, 3]) == (0b101, 0b1100, 1)


@pytest.mark.parametrize(
    "n,gates",
    [
        (0, []),
        (21, []),
        (3, [("dense", [3], np.eye(2))]),
        (3, [("dense", [1, 1], np.eye(4))]),
        (6, [("dense", [0, 1, 2, 3, 4], np.eye(32))]),
        (3, [("CZ", [0], None)]),
    ],
)
def test_add_circuit_rejects_bad_input(n, gates):
    b = Batch()
    with pytest.raises(QulacsMI355Error):
        b.add(n, gates, [])
    assert len(b) == 0


def test_term_beyond_qubits_rejected():
    b = Batch()
    with pytest.raises(QulacsMI355Error):
        b.add(3, [], [(1 << 3, 0, 0, 1.0)])


def test_compile_argument_checks_before_device_work():
    b = Batch()
    b.add(5, [("dense", [0, 1, 2, 3], np.eye(16))], [])
    with pytest.raises(QulacsMI355Error):
        b.compile(block_qubits=3)  # 4-qubit gate needs a 4-qubit block
    with pytest.raises(QulacsMI355Error):
        b.compile(block_qubits=5)


def test_fused_circuit_rejects_bad_arguments():
    from qulacs_amd.batch import FusedCircuit

    with pytest.raises(QulacsMI355Error):
        FusedCircuit(3, [])  # below 4 qubits
    with pytest.raises(QulacsMI355Error):
        FusedCircuit(10, [], local_qubits=7)
    with pytest.raises(QulacsMI355Error):
        FusedCircuit(10, [("dense", [0, 1, 2], np.eye(8))], block_qubits=2)
    fc = FusedCircuit(24, [("dense", [q], np.eye(2)) for q in range(24)] + [("CZ", [0, 23], None)])
    st = fc.stats()
    assert st["stages"] >= 2 and st["passes"] >= st["stages"]
    fc.close()


def test_fused_defaults():
    """Width and window 0 pick 3-qubit blocks and 12-qubit windows, and 4 and 13 from 20 qubits on where
    that saves a stage of a circuit with at most two operations a qubit; a 4-qubit dense gate
    widens the default block."""
    from qulacs_amd.batch import FusedCircuit

    def stats(n, gates, **kw):
        fc = FusedCircuit(n, gates, **kw)
        try:
            return fc.stats()
        finally:
            fc.close()

    def layer(n):  # 2 n - 1 operations
        return [("dense", [q], np.eye(2)) for q in range(n)] + [("CZ", [q, q + 1], None) for q in range(n - 1)]

    def ladder(n):  # 3 n - 3 operations
        return [("CNOT", [q, q + 1], None) for q in range(n - 1)]

    spread = [("dense", [q], np.eye(2)) for q in (3, 6, 9, 11, 13, 14, 16, 17, 18, 19)]
    narrow, wide = dict(block_qubits=3, local_qubits=12), dict(block_qubits=4, local_qubits=13)
    for n, gates, kw in [(8, layer(8), narrow), (13, layer(13), narrow), (16, layer(16), narrow),
                         (19, spread[:-1], narrow),  # a stage saved, but below 20 qubits
                         (20, layer(20), narrow), (21, layer(21), narrow),  # no stage saved
                         (20, spread, wide), (24, spread, wide), (22, layer(22), wide),
                         (22, 2 * layer(22), narrow), (23, ladder(23), narrow),  # too much arithmetic
                         (24, [("dense", [q, q + 1, q + 2], np.eye(8)) for q in range(20)], narrow)]:
        assert stats(n, gates) == stats(n, gates, **kw), (n, len(gates))
    for n, gates in [(20, spread), (22, layer(22)), (23, ladder(23))]:
        assert stats(n, gates, **wide)["stages"] < stats(n, gates, **narrow)["stages"]
    four = [("dense", [q], np.eye(2)) for q in range(16)] + [("dense", [1, 5, 9, 14], np.eye(16))]
    assert stats(16, four) == stats(16, four, block_qubits=4, local_qubits=12)


def test_server_rejects_bad_configuration():
    from qulacs_amd.serving import Server

    with pytest.raises(QulacsMI355Error):
        Server(hbm_budget_bytes=100)
    with pytest.raises(QulacsMI355Error):
        Server(hbm_budget_bytes=1 << 30, large_slots=0)
    with pytest.raises(QulacsMI355Error):
        Server(hbm_budget_bytes=1 << 30, small_max_qubits=17)


def test_adjoint_circuit_validation_is_host_only():
    from qulacs_amd.adjoint import AdjointCircuit, hardware_efficient_ansatz, heisenberg_terms

    gates, P = hardware_efficient_ansatz(20, 12)
    assert P == 480 and len(heisenberg_terms(20)) == 57
    c = AdjointCircuit(20, gates, P)
    c.close()
    with pytest.raises(QulacsMI355Error):
        AdjointCircuit(3, [("rot", [0], [4], 0, 1.0)], 1)  # Pauli id 4


def test_adjoint_create_is_linear_in_parameters():
    """60000 rotations, each with a parameter of its own: 4 ms, where 60000^2 comparisons of
    parameters with rotations take more than a second."""
    import time

    from qulacs_amd import _lib

    count = 60000
    arr = (_lib.QmAdjointGate * count)()
    for i in range(count):
        arr[i].kind, arr[i].qubit_count, arr[i].param, arr[i].coef = _lib.ADJ_ROT, 1, i, 1.0
        arr[i].qubits[0], arr[i].paulis[0] = i % 20, 1 + i // 20 % 3
    best = 1e9
    for _ in range(3):
        t0 = time.perf_counter()
        h = _lib.call("qm_adjoint_create", 20, arr, count, count)
        best = min(best, time.perf_counter() - t0)
        _lib.call("qm_adjoint_destroy", h)
    print(best, flush=True)
    assert best < 0.3


def test_adjoint_workspace_does_not_hold_every_partial_sum():
    """40000 parameters at 20 qubits: two states of 16 MiB, the matrices of the operations (64 bytes
    each, forward and backward), 24 bytes per parameter and three sums per operation, and at most
    12 MiB of partial sums."""
    pytest.importorskip("torch")
    from qulacs_amd import _lib
    from qulacs_amd.adjoint import AdjointCircuit, hardware_efficient_ansatz

    gates, params = hardware_efficient_ansatz(20, 1000)
    c = AdjointCircuit(20, gates, params)
    ops = params // 2
    fixed = 2 * (16 << 20) + 2 * 64 * ops + 24 * params + 24 * ops
    assert params == 40000
    assert fixed <= _lib.call("qm_adjoint_workspace_bytes", c.h, 1) <= fixed + (12 << 20)
    c.close()


def test_batch_window_setter_validation():
    from qulacs_amd import _lib

    b = Batch()
    with pytest.raises(QulacsMI355Error):
        _lib.call("qm_batch_set_local_qubits", b.h, 7)
    with pytest.raises(QulacsMI355Error):
        _lib.call("qm_batch_set_local_qubits", b.h, 14)
    _lib.call("qm_batch_set_local_qubits", b.h, 11)
    b.close()


@pytest.mark.parametrize("windows,run", [(None, [11, 12]), ((12, 13), [12]), ((13,), [12]), ((9, 13, 12, 9), [9, 12])])
def test_autotune_times_each_program_once(monkeypatch, windows, run):
    """A window above the widest that a batch runs is that one: not compiled and timed beside it,
    and not reported as a choice."""
    b = Batch()
    compiled = []
    monkeypatch.setattr(b, "compile", lambda k, keep, lq: compiled.append((k, lq)))
    monkeypatch.setattr(b, "run", lambda: None)
    times = b.autotune((3, 4), repeats=1, **({} if windows is None else {"local_candidates": windows}))
    want = [(k, lq) for k in (3, 4) for lq in run]
    assert list(times) == want and compiled[:-1] == want and compiled[-1] in want
    b.close()


def test_adjoint_pass_plan():
    """Stages (launches) and passes of the adjoint's sweeps, planned on the host: the 20-qubit, 12-layer
    hardware-efficient ansatz (480 rotations, two merged per qubit and layer, 228 CZ) runs in 7
    forward and 8 backward stages of some 6 passes; a Pauli string is one rotation between CZ gates,
    and what stands before the first rotation is not swept backwards."""
    pytest.importorskip("torch")
    from qulacs_amd.adjoint import AdjointCircuit, hardware_efficient_ansatz

    gates, P = hardware_efficient_ansatz(20, 12)
    st = AdjointCircuit(20, gates, P).stats()
    assert st["gates"] == 708 and st["passes"] == st["forward"][1] + st["backward"][1]
    assert st["forward"][0] <= 7 and st["forward"][1] <= 47, st
    assert st["backward"][0] <= 8 and st["backward"][1] <= 49, st
    wide = AdjointCircuit(6, [("rot", [0, 1, 2, 3], [1, 2, 1, 1], 0, 1.0)], 1).stats()
    assert wide == {"passes": 6, "gates": 1, "forward": (1, 3), "backward": (1, 3)}
    zrot = AdjointCircuit(6, [("rot", [0, 1, 2, 3], [3, 3, 3, 3], 0, 1.0), ("CZ", [0, 5], None)], 1).stats()
    assert zrot["forward"] == zrot["backward"] == (1, 1)
    fixed = AdjointCircuit(14, [("CNOT", [q, q + 1], None) for q in range(13)], 0).stats()
    assert fixed["forward"][0] >= 2 and fixed["backward"] == (0, 0)
