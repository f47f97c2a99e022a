"""The exact CDF over several work-groups against the sequential sum it stands for, bit for bit:
states whose chunks (4096 entries) are plain, hold ties, cross binades, are zero, mix all of
these, or stop being finite, in one window of the walk (1024 chunks) and across windows."""
from __future__ import annotations

import numpy as np
import pytest

from qulacs_amd import _lib
from tests.gpu_util import DevState

pytestmark = pytest.mark.gpu


def _amplitudes(kind, dim, rng):
    i = np.arange(dim)
    if kind == "random":
        a = rng.standard_normal(dim)
    elif kind == "uniform":  # every increment the same: long stretches with ties, crossings on chunk edges
        return np.full(dim, np.sqrt(1.0 / dim))
    elif kind == "few":  # few distinct values, sums that stop half-way between two grid points
        return np.array([2.0 ** -9, 2.0 ** -10, 3 * 2.0 ** -12, 0.0])[rng.integers(0, 4, dim)] * (1 + (i >= dim // 3) * 2.0 ** -26)
    elif kind == "growing":  # a crossing every few chunks, several in some
        a = np.exp2(12.0 * i / dim) * rng.standard_normal(dim)
    elif kind == "steep":
        a = np.exp2(-300.0 + 300.0 * i / dim)
    elif kind == "zeros":
        a = np.where((i // 5000) % 3 == 1, rng.standard_normal(dim), 0.0)
    elif kind == "late":  # zero up to the last chunk
        a = np.where(i >= dim - 700, 1.0, 0.0)
    elif kind == "tiny":  # sums among the subnormals, then a jump
        a = np.where(i < dim // 2, 2.0 ** -537 * rng.integers(0, 3, dim), 2.0 ** -500 * rng.standard_normal(dim))
        return a
    elif kind == "inf":
        a = rng.standard_normal(dim)
        a[dim // 2 + 77] = np.inf
        return a
    return a / np.sqrt(np.sum(a * a))


@pytest.mark.parametrize("n", [16, 17, 19, 22, 23])
@pytest.mark.parametrize("kind", ["random", "uniform", "few", "growing", "steep", "zeros", "late", "tiny", "inf"])
def test_same_bits(n, kind):
    dim = 1 << n
    a = _amplitudes(kind, dim, np.random.default_rng(n))
    want = np.concatenate([[0.0], np.add.accumulate(a * a)])  # real amplitudes: p = a * a, rounded once
    out = np.zeros(dim + 1)
    with DevState.from_host(a.astype(np.complex128)) as s:
        _lib.call("qm_sampling_cdf_host", out.ctypes.data_as(_lib.PD), s.ptr, dim, None, 0)
    print(n, kind, flush=True)
    bad = np.flatnonzero(out.view(np.uint64) != want.view(np.uint64))
    assert bad.size == 0, (bad[:4], out[bad[:4]], want[bad[:4]])
