"""GPU tests of the vectors of rank-deficient matrices: singular values of the
rounding level, of which several share a block of the bidiagonal with the large
ones.

The bidiagonals are LAPACK's dgebrd of the matrices.  Values whose relative gap
in sigma^2 is just above 1e-6 get vectors of their own, accurate to
eps / 1e-6 = 2e-10; 1e-9 leaves room for a handful of such pairs.
"""
import numpy as np
import pytest

from conftest import gpu_case

pytestmark = pytest.mark.gpu


def _check(ddcsvd, po, A):
    _, a, b, _, _ = po.lapack_dgebrd(np.asfortranarray(A))
    s, X, Y = ddcsvd.bdsvd_vectors(a, b)
    eye = np.eye(len(a))
    assert np.linalg.norm(X.T @ X - eye) <= 1e-9
    assert np.linalg.norm(Y.T @ Y - eye) <= 1e-9
    B = np.diag(a) + np.diag(b, 1)
    assert np.linalg.norm(B @ X - Y * s) <= 1e-12 * np.linalg.norm(B)


@pytest.mark.parametrize("seed", [0, 1, 2, 146, 147, 169, 170])
@pytest.mark.parametrize("kind", ["normal", "binary"])
def test_products_of_low_rank(ddcsvd, po, kind, seed):
    rng = np.random.default_rng(seed)
    n = int(rng.integers(20, 300))
    m, k = n + int(rng.integers(0, 100)), int(rng.integers(1, n))
    gpu_case(f"rank deficient {kind} {m} x {n} rank {k} seed {seed}")
    if kind == "normal":
        A = rng.standard_normal((m, k)) @ rng.standard_normal((k, n))
    else:
        A = (rng.integers(0, 2, (m, k)) @ rng.integers(0, 2, (k, n))).astype(float)
    _check(ddcsvd, po, A)


@pytest.mark.parametrize("seed", [2, 3, 23, 29, 31, 32, 63, 68, 80, 84, 114])
def test_zeros_beside_values_of_the_rounding_level(ddcsvd, po, seed):
    """A third of the rows and columns zero and one column twice: the bidiagonal
    holds exact zeros next to values down to eps^2 of the largest."""
    rng = np.random.default_rng(seed)
    n = int(rng.integers(20, 300))
    m = n + int(rng.integers(0, 100))
    gpu_case(f"rank deficient, zero rows and columns {m} x {n} seed {seed}")
    rng.integers(1, n)
    A = rng.standard_normal((m, n))
    A[:, rng.permutation(n)[:n // 3]] = 0
    A[:, n // 2] = A[:, 0]
    A[rng.permutation(m)[:m // 3]] = 0
    _check(ddcsvd, po, A)


@pytest.mark.parametrize("seed,m,n", [(40, 1455, 1451), (81, 773, 766), (129, 725, 688),
                                      (168, 560, 538), (236, 1981, 1792)])
@pytest.mark.parametrize("decades", [8, 12, 16])
def test_graded_columns(ddcsvd, seed, m, n, decades):
    """Columns falling to 10^-decades of the first: values on both sides of the
    rounding level in one block, many of them close.  The bound is that of above."""
    torch = pytest.importorskip("torch")
    gpu_case(f"graded columns {m} x {n} by 1e-{decades}")
    g = torch.Generator(device="cuda").manual_seed(seed)
    A = torch.randn(m, n, dtype=torch.float64, device="cuda", generator=g)
    A = A * torch.logspace(0, -decades, n, dtype=torch.float64, device="cuda")
    s, U, V = ddcsvd.svd_torch(A)
    eye = torch.eye(n, dtype=torch.float64, device="cuda")
    assert torch.linalg.norm(U.T @ U - eye) <= 1e-9
    assert torch.linalg.norm(V.T @ V - eye) <= 1e-9
    assert torch.linalg.norm((U * s) @ V.T - A) <= 1e-12 * torch.linalg.norm(A)
