"""qm_observable_expectation_host over the forms its grouping of terms meets: fewer
amplitudes than a coset (1..3 qubits), one block, several blocks, masks that depend on each
other, only Z strings, low pivots, more terms than the kernel arguments hold, groups
split over work-groups.

Tolerance: sums of 2^n products of magnitude |psi|^2, each rounded a few times:
|d| <= 2^-53 * (16 + 2 log2(2^n)) * sum |c_k| for a normalised state."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from qulacs_amd import _lib
from qulacs_amd.batch import pauli_masks
from tests.gpu_util import DevState, to_complex

pytestmark = pytest.mark.gpu


def _call(name, terms, s):
    k = len(terms)
    bf = (C.c_ulonglong * k)(*[t[0] for t in terms])
    pf = (C.c_ulonglong * k)(*[t[1] for t in terms])
    rot = (C.c_uint * k)(*[t[2] for t in terms])
    co = (_lib.QmComplex * k)(*[_lib.QmComplex(t[3].real, t[3].imag) for t in terms])
    return to_complex(_lib.call(name, bf, pf, rot, co, k, s.ptr, s.dim, None, 0))


def _parity(x, mask):
    v = (x & np.uint64(mask)).copy()
    for sh in (32, 16, 8, 4, 2, 1):
        v ^= v >> np.uint64(sh)
    return (v & np.uint64(1)).astype(np.int64)


def _want(terms, psi):
    x = np.arange(psi.size, dtype=np.uint64)
    e = 0.0
    for bf, pf, rot, c in terms:
        y = x ^ np.uint64(bf)
        e += c * np.vdot(psi, (1j ** rot) * (1 - 2 * _parity(y, pf)) * psi[y.astype(np.int64)]).real
    return e


def _terms(rng, n, kind, count):
    out = []
    for _ in range(count):
        if kind == "z":
            p = rng.choice([0, 3], n)
        elif kind == "low":
            p = np.zeros(n, dtype=int)
            p[:min(n, 5)] = rng.integers(0, 4, min(n, 5))
        elif kind == "pairs":  # X_i X_j, Y_i Y_j, Z_i Z_j: masks shared and dependent
            p = np.zeros(n, dtype=int)
            i = int(rng.integers(n))
            p[[i, (i + 1) % n]] = int(rng.integers(1, 4))
        else:
            p = rng.integers(0, 4, n)
        out.append((*pauli_masks(range(n), p), complex(rng.standard_normal(), rng.standard_normal())))
    return out


@pytest.mark.parametrize("n,kind,count", [(1, "any", 5), (2, "any", 9), (3, "any", 20), (4, "any", 30), (5, "pairs", 40),
                                          (9, "any", 1), (10, "z", 6), (13, "any", 24), (14, "low", 24), (14, "any", 24),
                                          (15, "pairs", 60), (16, "any", 130), (12, "any", 1200), (18, "any", 17)])
def test_observable_groups(n, kind, count):
    rng = np.random.default_rng(10 * n + count)
    psi = rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)
    psi /= np.linalg.norm(psi)
    terms = _terms(rng, n, kind, count)
    tol = 2.0 ** -53 * (16 + 2 * n) * sum(abs(t[3]) for t in terms)
    with DevState.from_host(psi) as s:
        got = _call("qm_observable_expectation_host", terms, s)
        assert abs(got - _want(terms, psi)) <= tol, (got, _want(terms, psi), tol)
        if count <= 128:
            assert _call("qm_observable_expectation_noalloc_host", terms, s) == got


@pytest.mark.parametrize("n,kind,count", [
    (2, "z", 200), (7, "any", 33), (10, "z", 32), (10, "z", 33), (10, "z", 49), (10, "any", 600), (11, "any", 8),
    (11, "z", 9), (12, "low", 300), (13, "any", 4), (13, "any", 5), (13, "z", 2000), (16, "z", 500), (20, "z", 100),
    (21, "z", 40)])
def test_groups_split_over_work_groups(n, kind, count):
    """Both sides of the rule for one block, groups split into pieces (all Z strings are one group),
    pieces among the kernel arguments and behind them.  Tolerance as above."""
    test_observable_groups(n, kind, count)


def test_infinities_and_nan_stay_where_they_were():
    """A NaN amplitude gives a NaN expectation; it does not hide behind a zero."""
    n = 6
    psi = np.full(1 << n, 2.0 ** -(n / 2), dtype=complex)
    psi[37] = np.nan
    with DevState.from_host(psi) as s:
        assert np.isnan(_call("qm_observable_expectation_host", [(1, 0, 0, 1.0 + 0j), (0, 3, 0, 1.0 + 0j)], s).real)
