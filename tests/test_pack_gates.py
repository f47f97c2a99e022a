"""Packing of gate lists for the C entry points: the compiled form against the gate-by-gate
conversion it replaces (reached with the compiled one switched off), over the containers, numbers
and matrix layouts that callers pass, and what is refused."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from qulacs_amd import _lib, batch

RNG = np.random.default_rng(5)


def _m(k):
    return RNG.standard_normal((1 << k, 1 << k)) + 1j * RNG.standard_normal((1 << k, 1 << k))


class _Int:
    def __int__(self):
        return 3


FORMS = {
    "plain": [("dense", [1], _m(1)), ("diag", [0, 2], np.exp(1j * RNG.uniform(0, 6, 4))), ("CZ", [0, 1], None),
              ("CNOT", (2, 1), None), ("dense", (0, 1, 2, 3), _m(4))],
    "empty": [],
    "layouts": [("dense", [0, 1], _m(2).T), ("dense", [0], _m(2)[::2, ::2]), ("dense", [0], np.asfortranarray(_m(1))),
                ("dense", [1], _m(1).real), ("dense", [1], [[0, 1], [1, 0]]), ("dense", [2], _m(1).astype(np.complex64)),
                ("dense", [3], _m(1).astype(">c16")), ("diag", [1], (1, 1j)),
                ("CZ", [0, 1], [1.0])],
    "numbers": [("CZ", [np.int64(1), np.uint8(2)], None), ("CZ", [1.0, True], None), ("CZ", ["2", _Int()], None),
                ("CZ", np.array([0, 1]), None), ("CZ", [-1, 2 ** 40 + 5], None)],
    "containers": [["CZ", [0, 1], None], np.array(["CZ", [0, 1], None], dtype=object), ("CZ", range(2), None)],
}


def _read(gates, monkeypatch, compiled):
    with monkeypatch.context() as m:
        if not compiled:
            m.setattr(batch._core, "_pack_gates", lambda *a: None)
        arr, keep = batch._marshal(gates)
    out = []
    for g, (kind, q, mat) in zip(arr, gates):
        size = 0 if mat is None else np.asarray(mat).size
        out.append((g.kind, g.qubit_count, list(g.qubits), bool(g.matrix),
                    C.string_at(C.cast(g.matrix, C.c_void_p), 16 * size) if size else b""))
    del keep
    return out


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("container", [list, tuple])
def test_same_as_gate_by_gate(form, container, monkeypatch):
    gates = container(FORMS[form])
    assert _read(gates, monkeypatch, True) == _read(gates, monkeypatch, False)


@pytest.mark.parametrize("bad", [("U", [0], None), ("CZ", [0, 1, 2, 3, 4], None), ("CZ", [0, None], None), ("CZ", 3, None),
                                 ([], [0], None), ("dense", [0], "x"), ("CZ", [0, 1]), 7, ("dense", [0], [[1, 2], [3]])])
def test_refused_alike(bad, monkeypatch):
    found = []
    for compiled in (True, False):
        with pytest.raises(Exception) as e, monkeypatch.context() as m:
            if not compiled:
                m.setattr(batch._core, "_pack_gates", lambda *a: None)
            batch._marshal([("CZ", [0, 1], None), bad])
        found.append((type(e.value), str(e.value)))
    assert found[0] == found[1]
    if isinstance(bad, tuple) and bad[0] == "U":
        assert found[0][0] is _lib.QulacsMI355Error
