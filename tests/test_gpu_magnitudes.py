"""GPU tests of the SVD of matrices and bidiagonals of any magnitude: the stages
work with products of squares of the singular values, whose range is left long
before that of the entries."""
import numpy as np
import pytest

from conftest import gpu_case
from ddcsvd import gen

pytestmark = pytest.mark.gpu

EXPS = [-900, -449, -400, -330, -280, -250, -150, -101, -100, -99, 99, 100, 101, 150, 250, 256, 330,
        400, 449, 900]


def _check(B, s, U, V):
    k = len(s)
    assert np.isfinite(s).all() and np.isfinite(U).all() and np.isfinite(V).all()
    ref = np.sort(np.linalg.svd(B, compute_uv=False))
    assert np.abs(s - ref).max() <= 1e-12 * ref[-1]
    assert np.linalg.norm(B - (U * s) @ V.T) <= 1e-12 * np.linalg.norm(B)
    assert np.linalg.norm(U.T @ U - np.eye(k)) <= 1e-10
    assert np.linalg.norm(V.T @ V - np.eye(k)) <= 1e-10


@pytest.mark.parametrize("p", EXPS)
@pytest.mark.parametrize("m,n", [(120, 100), (12, 208), (227, 5)])
def test_svd(ddcsvd, m, n, p):
    gpu_case(f"svd_gpu {m} x {n} at 2^{p}")
    A = gen.normal_matrix(m, n, 7)
    s, U, V, _ = ddcsvd.svd(np.ldexp(A, p))
    _check(A, np.ldexp(s, -p), U, V)


@pytest.mark.parametrize("p", EXPS)
def test_bidiagonal(ddcsvd, p):
    gpu_case(f"bdsvd_vectors at 2^{p}")
    rng = np.random.default_rng(11)
    a, b = rng.uniform(0.1, 1, 64), rng.uniform(-1, 1, 63)
    s, X, Y = ddcsvd.bdsvd_vectors(np.ldexp(a, p), np.ldexp(b, p))
    _check(np.diag(a) + np.diag(b, 1), np.ldexp(s, -p), Y, X)
    v = ddcsvd.bdsvd_values(np.ldexp(a, p), np.ldexp(b, p))
    assert np.abs(np.ldexp(v, -p) - np.ldexp(s, -p)).max() <= 1e-12
