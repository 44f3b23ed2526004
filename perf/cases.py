"""The workloads this library's speed is measured on.

A case is a dict of plain values; ``prepare`` makes what a program holds before
the call (inputs on the GPU, or host arrays for the drop-in entry points, and
the plan of a batch), ``run`` is one pass through the package's public entry
points, ``work`` the bytes and operations the pass cannot do without, and
``exact`` the same outputs from LAPACK in 64 bits.

Singular vectors are defined up to the sign of each pair.  The programs here
fix it as one that stores or compares factors does: the first row of U is made
non-negative, and V follows.

Kinds:
  svd      ddcsvd.svd_torch on a dense FP64 CUDA matrix (svd_gpu_dev)
  host     ddcsvd.svd on a host array (the svd_gpu drop-in; A comes back
           holding the reflectors)
  bidiag   ddcsvd.bidiag on a host array (the bidiag_par drop-in)
  grad     forward and backward through ddcsvd.autograd.svd
  mixed    ddcsvd.svd_mixed_torch, FP32 updates and two refinement steps, on a
           spectrum without long runs of close values
  batched  BatchedSvd.run: a kept plan, one launch per pass
  noalloc  BatchedSvd.run_noalloc: the entry point without device allocation
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "ddc-svd_amd"))

import ddcsvd  # noqa: E402
import ddcsvd.autograd  # noqa: E402
from ddcsvd import batched, gen  # noqa: E402

F64 = torch.float64
DTYPES = {"f64": torch.float64, "f32": torch.float32}


def listed():
    return [
        # one small dense matrix at a time, where launches and latency count
        {"name": "svd_96x64", "kind": "svd", "m": 96, "n": 64, "dist": "uniform"},
        # the reference's own smoke size, entries U(-1, 1)
        {"name": "svd_512x256", "kind": "svd", "m": 512, "n": 256, "dist": "uniform"},
        # an ordinary matrix of odd sizes (no dimension a multiple of a tile)
        {"name": "svd_1531x1187", "kind": "svd", "m": 1531, "n": 1187, "dist": "normal"},
        # more columns than rows: the transposed layout
        {"name": "svd_1000x3000", "kind": "svd", "m": 1000, "n": 3000, "dist": "normal"},
        # the headline problem
        {"name": "svd_8192x8192", "kind": "svd", "m": 8192, "n": 8192, "dist": "normal"},
        # a C caller's call: host buffers in and out
        {"name": "host_640x480", "kind": "host", "m": 640, "n": 480, "dist": "uniform"},
        # stand-alone bidiagonalization of a host matrix
        {"name": "bidiag_2048x1536", "kind": "bidiag", "m": 2048, "n": 1536, "dist": "normal"},
        # differentiating through the SVD (a training step's forward and backward)
        {"name": "grad_2048x1024", "kind": "grad", "m": 2048, "n": 1024},
        # mixed precision with refinement to FP64 accuracy
        {"name": "mixed_3072", "kind": "mixed", "n": 3072},
        # the batched headline: ten thousand uneven matrices in one launch
        {"name": "batched_f64_10000", "kind": "batched", "count": 10000, "lo": 16, "hi": 256,
         "dtype": "f64"},
        # the same shapes in FP32, a quarter of them
        {"name": "batched_f32_2500", "kind": "batched", "count": 2500, "lo": 16, "hi": 256,
         "dtype": "f32"},
        # a few hundred small matrices from a caller that may not allocate
        {"name": "noalloc_f64_300", "kind": "noalloc", "count": 300, "lo": 8, "hi": 64,
         "dtype": "f64"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["svd", "svd", "svd", "host", "bidiag", "grad", "mixed", "batched",
                       "batched", "noalloc"])
    if kind == "svd":
        return {"kind": kind, "m": _log_int(rng, 40, 8192), "n": _log_int(rng, 40, 8192),
                "dist": rng.choice(["uniform", "normal"])}
    if kind in ("host", "bidiag"):
        return {"kind": kind, "m": _log_int(rng, 64, 2048), "n": _log_int(rng, 64, 2048),
                "dist": rng.choice(["uniform", "normal"])}
    if kind == "grad":
        m = _log_int(rng, 128, 2048)
        return {"kind": kind, "m": m, "n": min(m, _log_int(rng, 64, 1024))}
    if kind == "mixed":
        return {"kind": kind, "n": _log_int(rng, 512, 4096)}
    hi = _log_int(rng, 24, 256)
    if kind == "batched":
        return {"kind": kind, "count": _log_int(rng, 64, 10000), "lo": rng.randint(4, 16),
                "hi": hi, "dtype": rng.choice(["f64", "f64", "f32"])}
    hi = min(hi, 96)
    return {"kind": kind, "count": _log_int(rng, 8, 300), "lo": rng.randint(4, 16), "hi": hi,
            "dtype": rng.choice(["f64", "f64", "f32"])}


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _dense(case, seed):
    """m x n CUDA matrix: i.i.d. N(0, 1) or U(-1, 1) entries."""
    g = _generator(seed)
    if case["dist"] == "normal":
        return torch.randn(case["m"], case["n"], dtype=F64, device="cuda", generator=g)
    return torch.rand(case["m"], case["n"], dtype=F64, device="cuda", generator=g) * 2 - 1


def _linear_spectrum(m, n, seed):
    """Q diag(linspace(1, 2, n)) P^T with random orthonormal Q and P."""
    g = _generator(seed)
    q, _ = torch.linalg.qr(torch.randn(m, n, dtype=F64, device="cuda", generator=g))
    p, _ = torch.linalg.qr(torch.randn(n, n, dtype=F64, device="cuda", generator=g))
    s = torch.linspace(1, 2, n, dtype=F64, device="cuda")
    return (q * s) @ p.t().contiguous()


def _shapes(case):
    """Shapes of a batch: m uniform in [lo, hi], n uniform in [lo / 2, m]; every
    seventh matrix is wide."""
    lo, hi = case["lo"], case["hi"]
    ms, ns = gen.batch_shapes(case["count"], seed=0, mlo=lo, mhi=hi, nlo=lo // 2)
    ms, ns = ms.copy(), ns.copy()
    ms[3::7], ns[3::7] = ns[3::7].copy(), ms[3::7].copy()
    return ms, ns


def _batch_input(case, total, seed):
    x = torch.rand(total, dtype=F64, device="cuda", generator=_generator(seed)) * 2 - 1
    return x.to(DTYPES[case["dtype"]])


def _grad_inputs(case, seed):
    m, n = case["m"], case["n"]
    g = _generator(seed + 7919)
    rnd = lambda *s: torch.randn(*s, dtype=F64, device="cuda", generator=g)  # noqa: E731
    return _linear_spectrum(m, n, seed), rnd(n), rnd(m, n), rnd(n, n)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "svd":
        return {"kind": kind, "A": _dense(case, seed)}
    if kind in ("host", "bidiag"):
        return {"kind": kind, "A": np.asfortranarray(_dense(case, seed).cpu().numpy())}
    if kind == "grad":
        A, gs, gU, gV = _grad_inputs(case, seed)
        return {"kind": kind, "A": A.requires_grad_(True), "cotangents": (gs, gU, gV)}
    if kind == "mixed":
        n = case["n"]
        return {"kind": kind, "A": _dense({"m": n, "n": n, "dist": "normal"}, seed)}
    ms, ns = _shapes(case)
    plan = batched.BatchedSvd(ms, ns, dtype=DTYPES[case["dtype"]])
    A = _batch_input(case, int(plan.offA[-1]), seed)
    S, U, V = plan.outputs()
    # column of every element of the packed U and V, and where each column of U starts
    mn = np.minimum(ms, ns)
    lenU, lenV = np.repeat(ms, mn), np.repeat(ns, mn)
    cols = torch.arange(len(lenU), dtype=torch.int32, device="cuda")
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    return {"kind": kind, "plan": plan, "A": A, "S": S, "U": U, "V": V,
            "first": dev(np.cumsum(lenU) - lenU),
            "colU": torch.repeat_interleave(cols, dev(lenU)),
            "colV": torch.repeat_interleave(cols, dev(lenV))}


# --------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------

def _sign(x):
    return 1.0 - 2.0 * (x < 0).to(x.dtype)


def run(state):
    kind, A = state["kind"], state["A"]
    if kind in ("svd", "mixed"):
        if kind == "svd":
            sigma, U, V = ddcsvd.svd_torch(A)
        else:
            sigma, U, V, _ = ddcsvd.svd_mixed_torch(A, "f32", refine_steps=2, separated=True)
        s = _sign(U[0])
        return sigma, U.mul_(s), V.mul_(s)
    if kind == "host":
        sigma, U, V, reflectors = ddcsvd.svd(A)
        s = np.where(U[0] < 0, -1.0, 1.0)
        U *= s
        V *= s
        return sigma, U, V, reflectors
    if kind == "bidiag":
        return ddcsvd.bidiag(A)
    if kind == "grad":
        gs, gU, gV = state["cotangents"]
        sigma, U, V = ddcsvd.autograd.svd(A)
        s = _sign(U.detach()[0])
        U, V = U * s, V * s
        (gA,) = torch.autograd.grad((sigma, U, V), A, (gs, gU, gV))
        return sigma.detach(), U.detach(), V.detach(), gA
    S, U, V = state["S"], state["U"], state["V"]
    if kind == "batched":
        state["plan"].run(A, S, U, V)
    else:
        state["plan"].run_noalloc(A, S, U, V)
    s = _sign(U[state["first"]])
    U.mul_(torch.index_select(s, 0, state["colU"]))
    V.mul_(torch.index_select(s, 0, state["colV"]))
    return S, U, V


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------

def _svd_work(m, n, size=8.0):
    """A read once; sigma and thin U, V written once.  Operations: the
    bidiagonalization (4 M N^2 - 4/3 N^3 for M >= N) and the reflectors
    applied to both sets of N vectors (4 M N^2 - 2 N^3 and 2 N^3)."""
    M, N = float(max(m, n)), float(min(m, n))
    nbytes = size * (M * N + N + M * N + N * N)
    bidiag = 4 * M * N * N - 4.0 / 3.0 * N ** 3
    back = 4 * M * N * N
    return nbytes, bidiag, back


def work(case):
    kind = case["kind"]
    if kind in ("batched", "noalloc"):
        size = 8.0 if case["dtype"] == "f64" else 4.0
        w = [_svd_work(int(m), int(n), size) for m, n in zip(*_shapes(case))]
        return {"bytes": sum(x[0] for x in w), "flops": sum(x[1] + x[2] for x in w)}
    m = case.get("m", case["n"])
    n = case["n"]
    nbytes, bidiag, back = _svd_work(m, n)
    if kind == "bidiag":
        return {"bytes": 16.0 * m * n, "flops": bidiag}
    if kind == "host":
        return {"bytes": nbytes + 8.0 * m * n, "flops": bidiag + back}
    if kind == "grad":  # U^T gU, V^T gV, the product with V^T, and U W
        extra = 2.0 * m * n * n * 3 + 2.0 * n ** 3
        return {"bytes": nbytes + 8.0 * (2 * m * n + n * n + n), "flops": bidiag + back + extra}
    return {"bytes": nbytes, "flops": bidiag + back}


# --------------------------------------------------------------------------
# the same in 64 bits, from LAPACK
# --------------------------------------------------------------------------

def _lapack(A):
    """(sigma ascending, U, V) with the first row of U non-negative."""
    U, s, Vt = np.linalg.svd(A, full_matrices=False)
    U, s, V = U[:, ::-1], s[::-1], Vt[::-1].T
    f = np.where(U[0] < 0, -1.0, 1.0)
    return np.ascontiguousarray(s), U * f, V * f


def exact(case, seed):
    kind = case["kind"]
    if kind == "bidiag":
        return None  # checked against the start's by the bound of 64-bit results
    if kind in ("batched", "noalloc"):
        ms, ns = _shapes(case)
        mn = np.minimum(ms, ns).astype(float)
        if float(np.sum(mn * mn * np.maximum(ms, ns))) > 2e9:
            return None  # thousands of LAPACK calls: minutes
        A = _batch_input(case, int(np.sum(ms * ns)), seed).double().cpu().numpy()
        out, at = ([], [], []), 0
        for m, n in zip(ms.tolist(), ns.tolist()):
            s, U, V = _lapack(A[at:at + m * n].reshape(n, m).T)
            at += m * n
            for o, x in zip(out, (s, U, V)):
                o.append(x.ravel(order="F"))
        return tuple(np.concatenate(o) for o in out)
    m, n = case.get("m", case["n"]), case["n"]
    if float(max(m, n)) * min(m, n) ** 2 > 5e10:
        return None  # over about ten seconds of LAPACK
    if kind == "grad":
        A, gs, gU, gV = (x.cpu().numpy() for x in _grad_inputs(case, seed))
        s, U, V = _lapack(A)
        d = s[None, :] ** 2 - s[:, None] ** 2
        np.fill_diagonal(d, np.inf)
        J, K = U.T @ gU, V.T @ gV
        W = (J - J.T) / d * s[None, :] + s[:, None] * ((K - K.T) / d)
        W += np.diag(gs) - J / s[None, :]
        return s, U, V, (U @ W + gU / s[None, :]) @ V.T
    if kind == "mixed":
        A = _dense({"m": n, "n": n, "dist": "normal"}, seed).cpu().numpy()
    else:
        A = _dense(case, seed).cpu().numpy()
    s, U, V = _lapack(A)
    return (s, U, V, None) if kind == "host" else (s, U, V)
