"""Request server (qm_server_*) on the GPU: every result equals the same
request run alone, the oracle agrees (energies within 1e-10 * sum |c|, samples
identical for the same uniforms), and admission keeps the footprint within the
budget."""
from __future__ import annotations

import ctypes as C
import threading

import numpy as np
import pytest

from qulacs_amd.batch import pauli_masks
from qulacs_amd.serving import Server
from qulacs_amd.workloads import haar_unitary, serving_requests
from tests.batch_util import oracle_run

pytestmark = pytest.mark.gpu


def _requests():
    rs = serving_requests(14, rate=1000.0, seed=11, n_range=(3, 22), depth_range=(2, 8), samples=300)
    # one of each path: tiny (padded to 4 qubits), batched, fused large
    return rs


def _run_all(srv, rs):
    ids = [srv.submit(r.n, r.gates, r.terms, r.uniforms) for r in rs]
    return [srv.wait(i) for i in ids]


def test_results_equal_alone_and_in_the_mix(oracle):
    rs = _requests()
    print("sizes", [r.n for r in rs], flush=True)
    with Server(hbm_budget_bytes=1 << 33, large_slots=3, small_max_qubits=16) as srv:
        mixed = _run_all(srv, rs)
        st = srv.stats()
        print("stats", st, flush=True)
        assert st["completed"] == len(rs) and st["failed"] == 0
    for r, (e, smp, lat) in zip(rs, mixed):
        with Server(hbm_budget_bytes=1 << 33, large_slots=1, small_max_qubits=16) as alone_srv:
            e1, s1, _ = _run_all(alone_srv, [r])[0]
        assert e == e1 and np.array_equal(smp, s1), r.n
        psi, want = oracle_run(oracle, r.n, r.gates, r.terms)
        scale = max(1.0, sum(abs(t[3]) for t in r.terms))
        assert abs(e - want) < 1e-10 * scale, (r.n, e, want)
        assert np.array_equal(smp, oracle.sampling(psi, r.uniforms)), r.n
        assert lat > 0


def test_admission_respects_budget_and_threads_submit():
    rs = serving_requests(24, rate=1000.0, seed=12, n_range=(14, 22), depth_range=(2, 6), samples=64)
    budget = (16 << 22) * 2  # room for two 22-qubit states
    out = {}
    with Server(hbm_budget_bytes=budget, large_slots=4, small_max_qubits=15) as srv:
        def client(chunk):
            for k, r in chunk:
                out[k] = srv.wait(srv.submit(r.n, r.gates, r.terms, r.uniforms))
        th = [threading.Thread(target=client, args=(list(enumerate(rs))[i::3],)) for i in range(3)]
        for t in th:
            t.start()
        for t in th:
            t.join()
        st = srv.stats()
    print("stats", st, flush=True)
    assert len(out) == len(rs) and st["failed"] == 0
    assert st["peak_bytes"] <= budget


def test_four_qubit_gates_beside_ordinary_requests(oracle):
    """A dense gate on four qubits needs another block width than the other small requests: all
    succeed, and the others' results are those of a server without it."""
    rs = serving_requests(12, rate=1000.0, seed=21, n_range=(5, 14), depth_range=(2, 5), samples=40)
    rng = np.random.default_rng(3)
    for k, n in ((2, 4), (5, 9), (9, 14)):
        q = [int(t) for t in rng.choice(n, 4, replace=False)]
        rs[k].n = n
        rs[k].gates = [("dense", [t], haar_unitary(rng, 1)) for t in range(n)] + [("dense", q, haar_unitary(rng, 4))]
        rs[k].terms = [(1, 1 << (n - 1), 0, 0.5), (0, 6, 0, 1.5)]
    with Server(hbm_budget_bytes=1 << 33, large_slots=1, small_max_qubits=16) as srv:
        got = _run_all(srv, rs)
        assert srv.stats()["failed"] == 0
    with Server(hbm_budget_bytes=1 << 33, large_slots=1, small_max_qubits=16) as srv:
        plain = _run_all(srv, [r for k, r in enumerate(rs) if k not in (2, 5, 9)])
    assert [g[0] for k, g in enumerate(got) if k not in (2, 5, 9)] == [p[0] for p in plain]
    for r, (e, smp, _) in zip(rs, got):
        psi, want = oracle_run(oracle, r.n, r.gates, r.terms)
        assert abs(e - want) < 1e-10 * max(1.0, sum(abs(t[3]) for t in r.terms)), r.n
        assert np.array_equal(smp, oracle.sampling(psi, r.uniforms)), r.n


@pytest.mark.parametrize("n,count", [(17, 3000), (18, 5000), (20, 4000)])
def test_observables_of_thousands_of_terms(n, count):
    """More flip masks than one launch's groups take.  A product state, whose Pauli strings have
    products as expectation values.  Tolerance: each string's value is exact to a few roundings per
    qubit and amplitude sum, |d| <= 2^-53 * 8 n * sum |c_k|."""
    rng = np.random.default_rng(n)
    gates, bloch = [], []
    for t in range(n):
        u = haar_unitary(rng, 1)
        gates.append(("dense", [t], u))
        a, b = u[0, 0], u[1, 0]
        bloch.append([1.0, 2 * (np.conj(a) * b).real, 2 * (np.conj(a) * b).imag, abs(a) ** 2 - abs(b) ** 2])
    terms, want, scale = [], 0.0, 0.0
    for _ in range(count):
        p = np.where(rng.random(n) < 0.5, rng.integers(0, 4, n), 0)
        c = float(rng.standard_normal())
        terms.append((*pauli_masks(range(n), [int(x) for x in p]), c))
        want += c * np.prod([bloch[t][p[t]] for t in range(n)])
        scale += abs(c)
    with Server(hbm_budget_bytes=1 << 30, large_slots=1, small_max_qubits=16) as srv:
        e, _, _ = srv.wait(srv.submit(n, gates, terms, [0.5]))
        few, _, _ = srv.wait(srv.submit(n, gates, terms[:1], [0.5]))
    print(n, e - want, scale, flush=True)
    assert abs(e - want) <= 2.0 ** -53 * 8 * n * scale
    k = terms[0]
    assert abs(few - k[3] * np.prod([bloch[t][(2 if k[1] >> t & 1 else 1) if k[0] >> t & 1 else 3 * (k[1] >> t & 1)]
                                     for t in range(n)])) <= 2.0 ** -53 * 8 * n * abs(k[3])


def test_invalid_requests_rejected():
    from qulacs_amd._lib import QulacsMI355Error

    with Server(hbm_budget_bytes=1 << 24, large_slots=1) as srv:
        with pytest.raises(QulacsMI355Error):
            srv.submit(21, [], [], [0.5])  # 32 MiB state over a 16 MiB budget
        with pytest.raises(QulacsMI355Error):
            srv.submit(5, [("dense", [7], np.eye(2))], [], [0.5])
        e, s, _ = srv.wait(srv.submit(5, [], [(0, 1, 0, 2.0)], [0.25, 0.75]))
        assert e == 2.0 and list(s) == [0, 0]


@pytest.mark.parametrize("n", [6, 17])
def test_density_matrix_gates_rejected(n):
    """QM_BATCH_DEPOL belongs to qm_circuit_create on density matrices: a request, batched (6 qubits)
    or alone (17), has a state vector."""
    from qulacs_amd import _lib

    z = (_lib.QmComplex * 1)(_lib.QmComplex(0.9, 0.05))
    g = (_lib.QmBatchGate * 1)()
    g[0].kind, g[0].qubit_count, g[0].matrix = _lib.BATCH_DEPOL, 2, z
    g[0].qubits[0], g[0].qubits[1] = 0, 3
    none = (C.c_ulonglong * 1)()
    with Server(hbm_budget_bytes=1 << 30, large_slots=1, small_max_qubits=16) as srv:
        with pytest.raises(_lib.QulacsMI355Error):
            _lib.call("qm_server_submit", srv.h, n, g, 1, none, none, (C.c_uint * 1)(), (C.c_double * 1)(), 0,
                      (C.c_double * 1)(0.5), 1)
        assert srv.stats()["admitted"] == 0
