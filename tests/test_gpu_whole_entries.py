"""GPU tests of the vectors of bidiagonals with small whole entries: zeros on the
diagonal and off it, repeated values, and shifts that meet eigenvalues of leading
blocks exactly.

Values whose relative gap in sigma^2 is just above 1e-6 get vectors of their own,
accurate to eps / 1e-6 = 2e-10; 1e-9 leaves room for a handful of such pairs.
"""
import numpy as np
import pytest

from conftest import gpu_case

pytestmark = pytest.mark.gpu


def _check(ddcsvd, a, b):
    a, b = np.asarray(a, float), np.asarray(b, float)
    s, X, Y = ddcsvd.bdsvd_vectors(a, b)
    B, eye = np.diag(a) + np.diag(b, 1), np.eye(len(a))
    assert np.abs(s - np.sort(np.linalg.svd(B, compute_uv=False))).max() <= 1e-12 * s[-1]
    assert np.linalg.norm(X.T @ X - eye) <= 1e-9
    assert np.linalg.norm(Y.T @ Y - eye) <= 1e-9
    assert np.linalg.norm(B @ X - Y * s) <= 1e-12 * np.linalg.norm(B)


@pytest.mark.parametrize("a,b", [
    ([-1, 0, 0], [-1, -1]), ([0, 0, -1], [-1, 2]), ([1, 1, 0, -1], [-1, -1, -2]),
    ([-1, 0, -2, -1], [1, -1, -2]), ([0, 0, -1, -1, 0], [1, 1, -2, -1]),
    ([2, -1, 2, 0, 0, 1], [1, 0, 1, -1, 1]), ([0, 0, 1, -1, -2, 1], [-1, 2, 0, 1, -2]),
    ([1, 0, 0, -2, -1, 0], [2, -1, 1, -1, 1]), ([-2, 1, -2, 2, 0, 0, -2], [2, 1, -1, 0, 2, 1]),
    ([-2, -2, 0, 0, -1, 1, -1], [-2, 2, -1, 2, 1, 1])])
def test_zeros_on_the_diagonal(ddcsvd, a, b):
    gpu_case(f"bdsvd_vectors {a} {b}")
    _check(ddcsvd, a, b)


@pytest.mark.parametrize("seed", range(24))
def test_random_whole_entries(ddcsvd, seed):
    rng = np.random.default_rng(seed)
    n = int(rng.integers(2, 600))
    gpu_case(f"bdsvd_vectors whole entries n {n} seed {seed}")
    _check(ddcsvd, rng.integers(-2, 3, n), rng.integers(-2, 3, n - 1))
