"""GPU test of the back-transformation's triangular factor (bt_tdiag and
bt_tmerge in backtrans.hip): blocks of every shape of its 16, 64 and doubled
tiles, whole and ragged.

Bound: the products of reflectors are exact to (m + n) u, and the vectors of
the bidiagonal that they are applied to carry u / gap for close values: 1e-10
covers the gaps of these matrices, as elsewhere.
"""
import numpy as np
import pytest

from conftest import gpu_case

pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 15, 17, 33, 63, 65, 66, 80, 127, 130, 191, 194, 255, 258, 321,
                               450, 511, 514, 577])
@pytest.mark.parametrize("extra", [0, 37])
def test_triangular_factor(ddcsvd, n, extra):
    m = n + extra
    A = np.asfortranarray(np.random.default_rng(n).standard_normal((m, n)))
    gpu_case(f"wyform {m}x{n}")
    s, U, V, _ = ddcsvd.svd(A)
    assert np.linalg.norm(U.T @ U - np.eye(n)) <= 1e-10
    assert np.linalg.norm(V.T @ V - np.eye(n)) <= 1e-10
    assert np.linalg.norm(A - (U * s) @ V.T) <= 1e-10 * np.linalg.norm(A)
