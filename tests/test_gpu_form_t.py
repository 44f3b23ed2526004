"""GPU test of the triangular factor of a block of reflectors (bt_tdiag and
bt_tmerge in backtrans.hip) by itself: T (I/2 + strict_upper(W^T W)) = I.

An inverse X of a triangular M formed block by block from products with inverted
blocks satisfies |X M - I| <= c n u |X| |M| |X| |M| entrywise with a constant of
a few units (Higham, Accuracy and Stability, section 14.2); c = 4, u = 2^-53.
"""
import ctypes

import numpy as np
import pytest

from conftest import gpu_case

pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# edges of the 16 x 16 and 64 x 64 blocks and of the joined pairs of 64, 128, 256
@pytest.mark.parametrize("nb", [1, 2, 15, 16, 17, 31, 33, 63, 64, 65, 79, 80, 81, 127, 128, 129, 191, 192,
                                193, 255, 256, 257, 320, 321, 383, 385, 447, 511, 512])
def test_inverse(ddcsvd, nb):
    rng = np.random.default_rng(nb)
    W = np.tril(rng.standard_normal((nb + 40, nb)))
    W /= np.linalg.norm(W, axis=0)
    G = np.asfortranarray(W.T @ W)
    T = np.full((nb, nb), np.nan, order="F")
    gpu_case(f"triangular factor nb={nb}")
    ptr = lambda x: ctypes.c_void_p(x.ctypes.data)  # noqa: E731
    ddcsvd._check(ddcsvd.load().ddc_test_form_t(nb, ptr(G), ptr(T)))
    assert np.all(np.tril(T, -1) == 0.0)
    M = np.eye(nb) / 2 + np.triu(G, 1)
    a = np.abs(T) @ np.abs(M)
    assert np.all(np.abs(T @ M - np.eye(nb)) <= 4 * nb * 2.0 ** -53 * (a @ a))
    # and W T W^T is the block: I - W T W^T = H_1 ... H_nb, orthogonal
    Q = np.eye(nb + 40) - W @ T @ W.T
    assert np.linalg.norm(Q.T @ Q - np.eye(nb + 40)) <= 12 * (2 * nb + 40) * nb * 2.0 ** -53
