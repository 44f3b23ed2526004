"""GPU tests of what happens where the work-groups of a bidiagonalization in
registers (resident.hip) do not come together: each of its launches in turn is
made to wait for one work-group more than its grid has, so that its bounded
wait ends and the panel kernels (bidiag.hip) go on from the step reached.  And
the panel kernels alone, at the sizes of their own edges, which the library's
calls do in registers.

Bounds: as in test_gpu_resident.py, c (m + n) u with c = 12 (Higham, Accuracy
and Stability, section 19.3), u = 2^-53, or 2^-24 where the matrix and the
reflectors are stored in FP32.
"""
import ctypes

import numpy as np
import pytest

from conftest import gpu_case
from ddcsvd import gen

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _bidiag(ddcsvd, A, dtype, resident=1, absent=-1):
    """(reflectors, alpha, beta), the step from which the launches gave up or -1, ms"""
    m, n = A.shape
    R = np.asfortranarray(A, dtype=dtype)
    if R is A:
        R = A.copy(order="F")
    alpha, beta = np.zeros(min(m, n)), np.zeros(n - 1 if m >= n else m)
    stopped, ms = ctypes.c_int(), ctypes.c_float()
    ptr = lambda x: ctypes.c_void_p(x.ctypes.data)  # noqa: E731
    ddcsvd._check(ddcsvd.load().ddc_test_bidiag(m, n, ptr(R), int(dtype == np.float32), ptr(alpha),
                                                ptr(beta), resident, absent, ctypes.byref(stopped),
                                                ctypes.byref(ms)))
    return (R, alpha, beta), stopped.value, ms.value


def _check(ddcsvd, A, out, dtype):
    m, n = A.shape
    R, alpha, beta = out
    bound = 12 * (m + n) * (2.0 ** -53 if dtype == np.float64 else 2.0 ** -24)
    k = min(m, n)
    B = np.zeros((k, n if m >= n else m + 1))
    B[np.arange(k), np.arange(k)] = alpha
    B[np.arange(len(beta)), np.arange(len(beta)) + 1] = beta
    want = np.linalg.svd(A, compute_uv=False)
    got = np.linalg.svd(B, compute_uv=False)
    assert np.max(np.abs(got - want)) <= bound * want[0]
    if m < n:
        return
    U = torch.from_numpy(ddcsvd.form_u(R.astype(np.float64))).cuda()[:, :n].contiguous()
    V = torch.from_numpy(ddcsvd.form_v(R.astype(np.float64))).cuda()
    At, Bt = torch.from_numpy(np.ascontiguousarray(A)).cuda(), torch.from_numpy(B).cuda()
    eye = torch.eye(n, dtype=torch.float64, device="cuda")
    assert torch.linalg.norm(At - (U @ Bt) @ V.t().contiguous()).item() \
        <= bound * torch.linalg.norm(At).item()
    assert torch.linalg.norm(U.t().contiguous() @ U - eye).item() <= bound * np.sqrt(n)
    assert torch.linalg.norm(V.t().contiguous() @ V - eye).item() <= bound * np.sqrt(n)


# (3100, 3090) has a panel before its first launch
@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("shape", [(160, 150), (300, 200), (700, 600), (1100, 1000), (600, 1500),
                                   (1030, 1500), (3100, 3090)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_each_launch_in_turn_gives_up(ddcsvd, shape, dtype):
    m, n = shape
    A = gen.normal_matrix(m, n, seed=m + n).astype(dtype).astype(np.float64)
    last = -1
    for launch in range(16):
        gpu_case(f"resident launch {launch} of {m}x{n} {dtype.__name__} gives up")
        out, stopped, _ = _bidiag(ddcsvd, A, dtype, absent=launch)
        if stopped < 0:  # no such launch, or one of a single work-group, which waits for none
            break
        assert stopped > last and stopped % 32 == 0 and stopped < min(m, n)
        _check(ddcsvd, A, out, dtype)
        last = stopped
    assert launch >= 1
    _check(ddcsvd, A, out, dtype)


@pytest.mark.parametrize("shape", [(400, 200), (700, 600)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_giving_up_is_quick(ddcsvd, shape):
    """The wait is bound to about 1 ms: the call takes that and the panel kernels'
    time, 10 ms left for everything else (the best of three).  400 x 200: the
    work-groups of one XCD, 700 x 600: of all."""
    A = gen.normal_matrix(*shape, seed=1)
    gpu_case(f"resident launch 0 of {shape[0]}x{shape[1]} gives up, timed")
    extra = min(_bidiag(ddcsvd, A, np.float64, absent=0)[2]
                - _bidiag(ddcsvd, A, np.float64, resident=0)[2] for _ in range(3))
    print(f"[giving-up] {shape}: {extra:.2f} ms beyond the panel kernels", flush=True)
    assert extra <= 10.0


# (70, 66): the panel boundary k = 64 is column n - 2; (2500, 200), (4200, 130):
# several chunks of rows in the GEMVs; (33, 33), (65, 90): one step past a panel
@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("shape", [(1, 1), (5, 1), (2, 2), (3, 2), (8, 3), (33, 33), (64, 64), (70, 66),
                                   (130, 97), (300, 300), (2500, 200), (4200, 130), (1, 5), (2, 3),
                                   (33, 100), (65, 90), (200, 700)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
def test_panel_kernels_alone(ddcsvd, shape, dtype):
    m, n = shape
    A = gen.normal_matrix(m, n, seed=3 * m + n).astype(dtype).astype(np.float64)
    gpu_case(f"panel kernels alone {m}x{n} {dtype.__name__}")
    out, stopped, _ = _bidiag(ddcsvd, A, dtype, resident=0)
    assert stopped == -1
    _check(ddcsvd, A, out, dtype)
