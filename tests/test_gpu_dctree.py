"""GPU tests of the values stage's recursion tree and secular roots (dc.hip):
sizes where the depths' ranges change (powers of two, one before, one after,
odd) with smooth, graded and split spectra.

Bound: a merge drops entries of at most 8 u' of its scale (u' = 2^-52) and
its roots are exact to the rounding of the secular sum, so each of the at most
log2 n + 1 merges above a value moves it by a modest multiple of 8 u' sigma_max
(4 here, for the entries dropped together), plus a few u' of the reference.
"""
import numpy as np
import pytest

from conftest import gpu_case

pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

EPS = 2.0 ** -52


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 6, 7, 8, 9, 15, 16, 17, 31, 33, 64, 127, 129, 257])
@pytest.mark.parametrize("kind", ["chi", "graded", "split", "constant"])
def test_values_tree(ddcsvd, n, kind):
    rng = np.random.default_rng(100 * n + len(kind))
    if kind == "chi":
        a = np.sqrt(rng.chisquare(np.arange(n, 0, -1)))
        b = np.sqrt(rng.chisquare(np.arange(n - 1, 0, -1))) if n > 1 else np.zeros(0)
    elif kind == "graded":
        a = 10.0 ** (-14.0 * np.arange(n) / n) * (1 + 0.1 * rng.standard_normal(n))
        b = 0.3 * a[:-1] * rng.standard_normal(n - 1)
    elif kind == "split":
        a = rng.standard_normal(n)
        b = np.where(np.arange(n - 1) % 3 == 2, 0.0, 1e-7 * rng.standard_normal(n - 1))
    else:
        a, b = np.ones(n), np.ones(n - 1)
    gpu_case(f"values tree n={n} {kind}")
    s = np.sort(ddcsvd.bdsvd_values(a, b))[::-1]
    ref = np.linalg.svd(np.diag(a) + np.diag(b, 1), compute_uv=False)
    assert np.abs(s - ref).max() <= (32 * (np.log2(n) + 1) + 16) * EPS * ref[0]
