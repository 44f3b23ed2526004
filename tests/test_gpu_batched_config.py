"""GPU tests that the launch configuration of the batched SVD is a question of
time alone: which matrices a whole workgroup takes, in FP64 and FP32 and at
every block width, and what the tuner picks from its timings, leave the results
the same bit for bit."""
import numpy as np
import pytest

from conftest import gpu_case
from ddcsvd import gen

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# column counts around multiples of the column blocks (2, 4, 8) and of the 8 and
# 12 blocks of a super-block, row counts around the register classes
NS = [1, 2, 7, 8, 9, 15, 16, 17, 23, 24, 25, 31, 32, 33, 47, 48, 49, 63, 64, 65, 95, 96, 97, 127,
      128, 129, 159, 160, 161, 193, 200, 255, 256]
MS = [min(256, n + d) for n, d in zip(NS, [0, 62, 57, 120, 0, 33, 0, 1, 80, 16, 15] * 3)]


def _run(b, A, **kw):
    S, U, V = b.outputs()
    b.run(A, S, U, V, **kw)
    torch.cuda.synchronize()
    return S, U, V


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("variant", [0, 1, 2, 3])
def test_threshold_leaves_the_bits(ddcsvd, dtype, variant):
    from ddcsvd.batched import BatchedSvd
    gpu_case(f"batched thresholds {dtype} variant {variant}")
    ms, ns = list(MS), list(NS)
    ms[5::7], ns[5::7] = ns[5::7], ms[5::7]  # some of them wide
    b = BatchedSvd(ms, ns, dtype)
    A = b.pack([gen.uniform_matrix(m, n, seed=17 * k) for k, (m, n) in enumerate(zip(ms, ns))])
    want = None
    for coop in (1, 40, 100, 257):
        b.set_config(variant, 1, coop)
        got = _run(b, A)
        want = want or got
        for x, y in zip(got, want):
            assert torch.equal(x, y), f"coop_nt {coop}"
    b.close()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("count,hi", [(300, 256), (3000, 64)])
def test_tuning_leaves_the_bits(ddcsvd, dtype, count, hi):
    """Two plans, each tuned by its own timings, and the second again, which finds
    the first one's choice; the block width goes by the sizes."""
    from ddcsvd.batched import BatchedSvd
    gpu_case(f"batched tuning {dtype} {count} up to {hi}")
    ms, ns = gen.batch_shapes(count, seed=3, mhi=hi)
    want, var = None, None
    for rep in range(3):
        b = BatchedSvd(ms, ns, dtype)
        A = torch.from_numpy(gen.uniform01(int(b.offA[-1]), 3) - 0.5).to("cuda", dtype)
        if rep < 2:
            b.tune(A, *b.outputs())
        got = _run(b, A)
        want, var = want or got, b.config()["variant"] if var is None else var
        assert b.config()["variant"] == var
        for x, y in zip(got, want):
            assert torch.equal(x, y), f"plan {rep}"
        b.close()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("count,m,n,variant", [
    (1, 8, 8, 1), (2000, 8, 8, 1), (300, 8, 128, 1), (500, 200, 8, 1), (2000, 9, 9, 0),
    (2000, 128, 20, 0)])
def test_few_columns_take_narrow_blocks(ddcsvd, dtype, count, m, n, variant):
    """In both types: a block of 8 leaves most of a matrix's waves nothing."""
    from ddcsvd.batched import BatchedSvd
    gpu_case(f"batched width {dtype} {count} of {m} x {n}")
    b = BatchedSvd([m] * count, [n] * count, dtype)
    A = torch.from_numpy(gen.uniform01(int(b.offA[-1]), 3) - 0.5).to("cuda", dtype)
    _run(b, A)
    assert b.config()["variant"] == variant
    b.close()
