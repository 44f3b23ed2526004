"""GPU tests of the FP64 rotation of the batched SVD (jrot in batched.hip):
columns whose squared norms and dot products are subnormal or close to it,
columns in the span of the others, and the accuracy of many rotations.

u = 2^-53, mt x mn the tall orientation.
"""
import numpy as np
import pytest

from conftest import gpu_case
from ddcsvd import gen

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

U53 = 2.0 ** -53
CONFIGS = [(v, c) for v in range(4) for c in (1, 257)]


def _run(mats, variant, coop):
    """[(sigma, U, V)], sweeps of a batch of FP64 matrices"""
    from ddcsvd.batched import BatchedSvd
    b = BatchedSvd([a.shape[0] for a in mats], [a.shape[1] for a in mats], torch.float64)
    b.set_config(variant, 1, coop)
    S, U, V = b.outputs()
    info = torch.zeros(b.count, dtype=torch.int32, device="cuda")
    b.run(b.pack(mats), S, U, V, info)
    torch.cuda.synchronize()
    out = [b.unpack(k, S, U, V) for k in range(b.count)]
    b.close()
    return out, info.cpu().numpy()


def _check(mats, out, tol):
    for k, (a, (s, u, v)) in enumerate(zip(mats, out)):
        mn = min(a.shape)
        name = f"matrix {k} {a.shape}"
        assert np.isfinite(s).all() and np.isfinite(u).all() and np.isfinite(v).all(), name
        t = tol(k, a)
        assert np.abs(u.T @ u - np.eye(mn)).max() <= t, name
        assert np.abs(v.T @ v - np.eye(mn)).max() <= t, name
        assert np.linalg.norm(a - (u * s) @ v.T) <= t * mn * np.linalg.norm(a), name


@pytest.mark.parametrize("variant,coop", CONFIGS)
def test_tiny_columns(ddcsvd, variant, coop):
    """Two columns of size t beside one of size 1, with equal and with unequal
    norms.  Their squared norms lose digits to the subnormal range: the working
    copy holds them as t / 2 or more, squared t^2 / 4, in multiples of 2^-1074;
    mt products per dot product and a rounding of each norm, 8 mt 2^-1074 / t^2
    together, beside the stopping test's mt u."""
    gpu_case(f"batched tiny columns variant {variant} coop {coop}")
    e = np.eye(4)
    mats, size = [], []
    for t in (1e-100, 1e-140, 1e-148, 1e-150, 1e-152, 1e-153, 1e-154, 1e-155, 1e-156, 1e-157,
              1e-158):
        mats += [np.stack([.5 * e[0], t * (e[1] + e[2] + e[3]), t * (e[1] + e[2] - e[3])], 1),
                 np.stack([.5 * e[0], t * (e[1] + e[2] + e[3]), t * (2 * e[1] + e[2] - e[3])], 1),
                 np.stack([e[0], t * e[1], t * (e[1] / 2 + e[2])], 1),
                 np.stack([e[0], t * e[1], t * e[1]], 1)]
        size += [t] * 4
    out, info = _run(mats, variant, coop)
    lost = 2.0 ** -537  # 2^-1074 / t^2 = (2^-537 / t)^2
    _check(mats, out, lambda k, a: 8 * 4 * ((lost / size[k]) ** 2 + U53))
    # squared norms with all their digits: converged
    assert (info[np.array(size) >= 1e-153] >= 1).all()


@pytest.mark.parametrize("variant,coop", CONFIGS)
def test_low_rank(ddcsvd, variant, coop):
    """Sums of one to three products of 0/1 vectors.  The columns beyond the
    rank shrink by u per rotation down to where squares underflow (2^-537, ten
    rotations) or where the sweeps end (info -1: those columns, of no
    consequence to A, are left as they are).  A matrix reported as converged has
    an orthonormal U; columns that ended in the range of the test above keep
    the digits that their size leaves them: sigma > 2^-500 sigma_max alone."""
    gpu_case(f"batched low rank variant {variant} coop {coop}")
    rng = np.random.default_rng(7)
    mats = []
    for k in range(200):
        m, n = int(rng.integers(8, 68)), int(rng.integers(8, 68))
        mats.append(sum(np.outer(rng.integers(0, 2, m), rng.integers(0, 2, n))
                        for _ in range(1 + k % 3)).astype(float))
    out, info = _run(mats, variant, coop)
    for k, (a, (s, u, v)) in enumerate(zip(mats, out)):
        mt, mn = max(a.shape), min(a.shape)
        name = f"matrix {k} {a.shape}"
        assert np.isfinite(s).all() and np.isfinite(u).all() and np.isfinite(v).all(), name
        big = s > 2.0 ** -500 * max(s[-1], 2.0 ** -500)
        y, z = (u, v) if a.shape[0] >= a.shape[1] else (v, u)
        t = 4 * np.sqrt(mt) * mn * U53
        if info[k] > 0:
            assert np.linalg.norm(y[:, big].T @ y[:, big] - np.eye(big.sum())) <= t, name
        assert np.linalg.norm(z.T @ z - np.eye(mn)) <= max(t, 1e-13 * mn), name
        assert np.linalg.norm(a - (u * s) @ v.T) <= 1e-13 * np.linalg.norm(a), name


@pytest.mark.parametrize("variant,coop", CONFIGS)
def test_sweeps_on_rank_one(ddcsvd, variant, coop):
    """A column parallel to another loses 53 bits to a rotation whose angle is
    exact to rounding, and 537 bits make its square zero: 11 rotations, one a
    sweep at least, and as many sweeps as a matrix without such columns takes
    (7) around them."""
    gpu_case(f"batched rank one variant {variant} coop {coop}")
    mats = [np.ones(s) for s in ((16, 8), (40, 33), (100, 64), (64, 100), (250, 200))]
    out, info = _run(mats, variant, coop)
    for a, (s, u, v) in zip(mats, out):
        assert np.linalg.norm(a - (u * s) @ v.T) <= 1e-13 * np.linalg.norm(a)
    assert (info >= 1).all() and (info <= 18).all(), info


@pytest.mark.parametrize("variant,coop", CONFIGS)
def test_rotations_do_not_drift(ddcsvd, variant, coop):
    """A column goes through at most 13 (mn - 1) rotations (13 sweeps, the most
    that random matrices of these sizes take).  Where cos^2 + sin^2 - 1 has no
    bias, each adds a random error of at most 2 u, together 2 u times the square
    root of their number; 4 covers the largest of all entries.  A bias would
    add up to its number."""
    gpu_case(f"batched drift variant {variant} coop {coop}")
    mats = [gen.uniform_matrix(m, n, seed=31 * m + n)
            for m, n in ((256, 256), (256, 200), (240, 256), (200, 180), (128, 120), (64, 60))]
    out, _ = _run(mats, variant, coop)
    for a, (s, u, v) in zip(mats, out):
        bound = 4 * U53 * np.sqrt(13.0 * (min(a.shape) - 1))
        ref = np.sort(np.linalg.svd(a, compute_uv=False))
        assert np.abs(s - ref).max() <= bound * ref[-1], a.shape
        assert np.linalg.norm(a - (u * s) @ v.T) <= bound * np.linalg.norm(a), a.shape
