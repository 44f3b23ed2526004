"""GPU tests of the bidiagonalization with the matrix in registers
(resident.hip): sizes at the limits of its kernel shapes and one past them, a
NaN with the bits of the exchange's empty mark, and a GPU whose CUs are held
by other work (the steps then run elsewhere).

Bounds: Householder transformations applied in floating point satisfy
||A - U B V^T||_F <= c (m + n) u ||A||_F and ||U^T U - I||_F, ||V^T V - I||_F
<= c (m + n) u sqrt(n) with a modest constant (Higham, Accuracy and Stability,
section 19.3); c = 12 here, u = 2^-53.
"""
import numpy as np
import pytest

from conftest import gpu_case
from ddcsvd import gen

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

U53 = 2.0 ** -53

# limits of the shapes, rows x columns: 128 x 64, 128 x 128, 256 x 256,
# 512 x 256, 512 x 512, 1024 x 512, 2048 x 512, 1024 x 1024, 4096 x 512,
# 2048 x 1024, 4096 x 1024, 2048 x 2048, 8192 x 512, 4096 x 2048
EDGES = [(128, 64), (129, 64), (128, 65), (128, 128), (129, 128), (256, 129), (256, 256),
         (257, 256), (512, 256), (512, 257), (512, 512), (513, 512), (1024, 512), (1025, 512),
         (1024, 513), (1024, 1024), (1025, 1024), (2048, 512), (2049, 130), (2048, 1024),
         (2049, 1025), (4097, 33)]


def _residual(ddcsvd, A):
    """(||A - U B V^T||_F / ||A||_F, ||U^T U - I||_F, ||V^T V - I||_F)"""
    m, n = A.shape
    R, alpha, beta = ddcsvd.bidiag(A)
    U = torch.from_numpy(ddcsvd.form_u(R)).cuda()[:, :n]
    V = torch.from_numpy(ddcsvd.form_v(R)).cuda()
    B = torch.diag(torch.from_numpy(alpha)) + torch.diag(torch.from_numpy(beta), 1) \
        if n > 1 else torch.from_numpy(alpha).reshape(1, 1)
    At = torch.from_numpy(np.ascontiguousarray(A)).cuda()
    res = (torch.linalg.norm(At - (U @ B.cuda()) @ V.t().contiguous())
           / torch.linalg.norm(At)).item()
    eye = torch.eye(n, dtype=torch.float64, device="cuda")
    return (res, torch.linalg.norm(U.t().contiguous() @ U - eye).item(),
            torch.linalg.norm(V.t().contiguous() @ V - eye).item())


@pytest.mark.parametrize("shape", EDGES, ids=lambda s: f"{s[0]}x{s[1]}")
def test_bidiag_at_the_limits_of_the_shapes(ddcsvd, shape):
    m, n = shape
    gpu_case(f"resident bidiag {m}x{n}")
    A = gen.normal_matrix(m, n, seed=m * 8209 + n)
    res, ou, ov = _residual(ddcsvd, A)
    assert res <= 12 * (m + n) * U53
    assert ou <= 12 * (m + n) * U53 * np.sqrt(n)
    assert ov <= 12 * (m + n) * U53 * np.sqrt(n)


@pytest.mark.parametrize("shape", [(4096, 2048), (8192, 513), (3072, 3072), (3200, 3104)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
def test_svd_dev_at_the_limits_of_the_large_shapes(ddcsvd, shape):
    m, n = shape
    gpu_case(f"resident svd {m}x{n}")
    g = torch.Generator(device="cuda").manual_seed(m + n)
    A = torch.randn(m, n, dtype=torch.float64, device="cuda", generator=g)
    s, U, V = ddcsvd.svd_torch(A)
    want = np.sort(np.linalg.svd(A.cpu().numpy(), compute_uv=False))
    assert np.max(np.abs(s.cpu().numpy() - want)) <= 12 * (m + n) * U53 * want[-1]
    # vectors of close values carry eps / gap: 1e-10 relative residual
    res = (torch.linalg.norm(A - (U * s) @ V.t().contiguous()) / torch.linalg.norm(A)).item()
    assert res <= 1e-10


@pytest.mark.parametrize("shape", [(65, 130), (300, 301), (511, 1100), (1030, 1500)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
def test_bidiag_wide_at_the_limits(ddcsvd, shape):
    m, n = shape
    gpu_case(f"resident wide bidiag {m}x{n}")
    A = gen.normal_matrix(m, n, seed=m * 8209 + n)
    _, alpha, beta = ddcsvd.bidiag(A)
    B = np.zeros((m, m + 1))
    B[np.arange(m), np.arange(m)] = alpha
    B[np.arange(m), np.arange(m) + 1] = beta
    want = np.linalg.svd(A, compute_uv=False)
    got = np.linalg.svd(B, compute_uv=False)
    assert np.max(np.abs(got - want)) <= 12 * (m + n) * U53 * want[0]


@pytest.mark.parametrize("shape", [(100, 60), (300, 200), (1100, 700)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
def test_bidiag_of_a_nan_with_all_bits_set_returns(ddcsvd, shape):
    m, n = shape
    gpu_case(f"resident bidiag with NaN {m}x{n}")
    A = gen.normal_matrix(m, n, seed=5)
    A[m // 2, n // 2] = np.array([2 ** 64 - 1], dtype=np.uint64).view(np.float64)[0]
    _, alpha, _ = ddcsvd.bidiag(A)
    assert np.isnan(alpha).any()


def test_svd_beside_work_that_holds_the_cus(ddcsvd):
    """A batched launch that fills the GPU for some tens of milliseconds runs
    on another stream: the work-groups of the resident kernel may not
    assemble, and the result is the same to rounding."""
    from ddcsvd import batched
    gpu_case("resident svd beside a batched launch")
    ms, ns = gen.batch_shapes(3000, seed=0)
    b = batched.BatchedSvd(ms, ns)
    b.set_config(0, 3, 32)
    A = torch.rand(int(b.offA[-1]), dtype=torch.float64, device="cuda") - 0.5
    out = b.outputs()
    X = torch.randn(700, 400, dtype=torch.float64, device="cuda")
    b.run(A, *out)
    alone = ddcsvd.svd_torch(X)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        b.run(A, *out)
    s, U, V = ddcsvd.svd_torch(X)
    torch.cuda.synchronize()
    assert torch.max(torch.abs(s - alone[0])).item() <= 12 * 1100 * U53 * s[-1].item()
    res = (torch.linalg.norm(X - (U * s) @ V.t().contiguous()) / torch.linalg.norm(X)).item()
    assert res <= 1e-12
    b.close()
