"""GPU tests of the two forms of the vectors' kernel (tw_solve in twisted.hip): with
one pair of waves per group of 64 values, which only matrices of more than 8192
columns take by themselves, and with two.  Both form every value by the same
operations in the same order, so they agree bit for bit; sizes around the 64
values of a group, the 64 entries of a chunk and odd and even numbers of chunks.
"""
import ctypes

import numpy as np
import pytest

from conftest import gpu_case

pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _vectors(ddcsvd, a, b, pairs):
    n = len(a)
    s, X, Y = np.zeros(n), np.zeros((n, n), order="F"), np.zeros((n, n), order="F")
    ptr = lambda x: ctypes.c_void_p(x.ctypes.data)  # noqa: E731
    ddcsvd._check(ddcsvd.load().ddc_test_vectors(n, ptr(a), ptr(b), ptr(s), ptr(X), ptr(Y), pairs))
    return s, X, Y


@pytest.mark.parametrize("n", [1, 2, 3, 63, 64, 65, 127, 128, 129, 191, 193, 257, 449, 1187])
@pytest.mark.parametrize("kind", ["chi", "graded", "split", "constant"])
def test_one_and_two_pairs_agree(ddcsvd, n, kind):
    rng = np.random.default_rng(10 * n + len(kind))
    if kind == "chi":
        a = np.sqrt(rng.chisquare(np.arange(n, 0, -1)))
        b = np.sqrt(rng.chisquare(np.arange(n - 1, 0, -1))) if n > 1 else np.zeros(0)
    elif kind == "graded":
        a = 10.0 ** (-12.0 * np.arange(n) / n) * (1 + 0.1 * rng.standard_normal(n))
        b = 0.3 * a[:-1] * rng.standard_normal(n - 1)
    elif kind == "split":  # blocks of three with close values
        a = 1.0 + rng.standard_normal(n) * 1e-7
        b = np.where(np.arange(n - 1) % 3 == 2, 0.0, 0.1 * rng.standard_normal(n - 1))
    else:
        a, b = np.ones(n), np.ones(n - 1)
    gpu_case(f"twisted pairs n={n} {kind}")
    one, two = (_vectors(ddcsvd, a, b, p) for p in (1, 2))
    for x, y in zip(one, two):
        assert np.isfinite(x).all()
        assert np.array_equal(x, y)
