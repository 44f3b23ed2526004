// backtrans.hip -- U = Q_left [Yb; 0], V = Q_right Xb on the FP64 matrix cores.
//
// Replaces multU / multV (bidiag_par.c:990-1095) and the per-vector OpenMP
// loop of svd_gpu.c:117-121, which apply the reflectors one vector at a
// time (BLAS1).  Here the reflectors stored in A are grouped into blocks of
// NBB and applied in compact WY form,
//     H_k0 ... H_{k0+NBB-1} = I - W T W^T,   T upper triangular,
// for the unit-norm convention H = I - 2 w w^T (tau = 2).  The inverse of T is
// T^{-1} = I/2 + strict_upper(W^T W) (the identity behind
// the recursive T-factor of LAPACK dlarft), so a block costs
//     G = W^T W,  Z = W^T C,  Z = T Z,  C -= W Z
// (in FP64 T is formed from G by bt_tdiag and bt_tmerge and applied as a
// product, elsewhere by a triangular solve with T^{-1})
// with the block's reflectors first packed into a dense zero-padded W; the
// three products are library GEMMs (rocBLAS, FP64 MFMA).
// Left reflectors are the columns A[k:m, k]; right reflectors are the rows
// A[k, k+1:n] (leading dimension n for V -- the reference indexes the
// transposed copy with m, bidiag_par.c:1034-1036, wrong when m != n).
#include <algorithm>

#include "ddc_common.h"

namespace ddc {

constexpr int NBB = 512;  // reflectors per compact-WY block

// C(0:n, 0:n) = Bt^T where Bt[j*ldb + i] holds vector i, entry j;
// rows n..rows-1 of C are zeroed.  TC: element type of C.
template <typename TC>
__global__ void bt_unpack(int n, int rows, const double* Bt, int ldb, TC* C, int ldc) {
  __shared__ double tile[32][33];
  int bx = blockIdx.x * 32, by = blockIdx.y * 32;  // bx: i (vector), by: j (entry)
  int tx = threadIdx.x, ty = threadIdx.y;          // 32 x 8
  for (int r = ty; r < 32; r += 8) {
    int j = by + r, i = bx + tx;
    tile[r][tx] = (j < n && i < n) ? Bt[(int64_t)j * ldb + i] : 0.0;
  }
  __syncthreads();
  // write C(j, i): consecutive threads take consecutive j (rows)
  for (int r = ty; r < 32; r += 8) {
    int i = bx + r, j = by + tx;
    if (i < n && j < rows) C[(int64_t)j + (int64_t)i * ldc] = (TC)((j < n) ? tile[tx][r] : 0.0);
  }
}

// D (c x r) = S^T for the r x c matrix S.
__global__ void k_transpose(int r, int c, const double* S, int lds, double* D, int ldd) {
  __shared__ double tile[32][33];
  int r0 = blockIdx.x * 32, c0 = blockIdx.y * 32;
  int tx = threadIdx.x, ty = threadIdx.y;
  for (int q = ty; q < 32; q += 8) {
    int i = r0 + tx, j = c0 + q;
    if (i < r && j < c) tile[q][tx] = S[(int64_t)i + (int64_t)j * lds];
  }
  __syncthreads();
  for (int q = ty; q < 32; q += 8) {
    int j = c0 + tx, i = r0 + q;
    if (i < r && j < c) D[(int64_t)j + (int64_t)i * ldd] = tile[tx][q];
  }
}

int transpose_f64(int r, int c, const double* S, int lds, double* D, int ldd, hipStream_t st) {
  if (r <= 0 || c <= 0) return DDC_OK;
  dim3 g((unsigned)ceil_div(r, 32), (unsigned)ceil_div(c, 32));
  hipLaunchKernelGGL(k_transpose, g, dim3(32, 8), 0, st, r, c, S, lds, D, ldd);
  DDC_LAUNCHED();
  return DDC_OK;
}

// Dense copy Wd (rows x nb, ld ldw) of a block of reflectors, zeros
// outside their support.  left: Wd(i, c) = A[k0+i, k0+c] for i >= c.
// right: Wd(i, c) = A[k0+c, k0+1+i] for i >= c (rows of A, read through an
// LDS tile so that both sides stay coalesced).
template <bool RIGHT, typename T>
__global__ void bt_pack(int rows, int nb, const T* S, int lda, T* Wd, int ldw) {
  __shared__ T tile[32][33];
  const int i0 = blockIdx.x * 32, c0 = blockIdx.y * 32;
  const int tx = threadIdx.x, ty = threadIdx.y;  // 32 x 8
  if (!RIGHT) {
    for (int q = ty; q < 32; q += 8) {
      const int i = i0 + tx, c = c0 + q;
      if (i < rows && c < nb) Wd[i + (int64_t)c * ldw] = i >= c ? S[i + (int64_t)c * lda] : T(0);
    }
  } else {
    for (int q = ty; q < 32; q += 8) {  // tile[c][i] = S(c, i), coalesced over c
      const int c = c0 + tx, i = i0 + q;
      tile[q][tx] = (c < nb && i < rows && i >= c) ? S[c + (int64_t)i * lda] : T(0);
    }
    __syncthreads();
    for (int q = ty; q < 32; q += 8) {
      const int i = i0 + tx, c = c0 + q;
      if (i < rows && c < nb) Wd[i + (int64_t)c * ldw] = tile[tx][q];
    }
  }
}

// T^{-1} = I/2 + strict_upper(G) (nb x nb, ld nb) for the block
// H_0 ... H_{nb-1} = I - W T W^T of unit-norm reflectors (tau = 2).
template <typename T>
__global__ void bt_tinv(int nb, const T* G, T* Ti) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= nb * nb) return;
  const int i = e % nb, j = e / nb;
  Ti[e] = i < j ? G[e] : (i == j ? T(0.5) : T(0));
}

// T (nb x nb, ld nb, zeros below the diagonal) from G = W^T W in two kernels:
// the 64 x 64 diagonal blocks of I/2 + strict_upper(G) are inverted in LDS
// (bt_tdiag), then ever larger pairs of inverted blocks are joined (bt_tmerge,
// one launch per doubling):
//     [A B; 0 C]^{-1} = [A^{-1}, -A^{-1} B C^{-1}; 0, C^{-1}].
// A block's chain of dependent launches is what it costs, not its arithmetic
// (a 512 x 512 T is 0.1 GFLOP): one to four launches instead of the 8 to 11 of
// the library's triangular inverse took the back-transformation from 0.25 to
// 0.13 ms at 96 x 64, 0.37 to 0.22 at 512 x 256 and 1.17 to 0.98 at
// 1531 x 1187.
constexpr int TB = 64;

__global__ __launch_bounds__(256) void bt_tdiag(int nb, const double* G, double* T) {
  const int tid = threadIdx.x;
  const int i0 = blockIdx.x * TB, j0 = blockIdx.y * TB;
  if (i0 < j0) return;
  if (i0 > j0) {
    for (int e = tid; e < TB * TB; e += 256) {
      const int i = i0 + e % TB, j = j0 + e / TB;
      if (i < nb && j < nb) T[i + (int64_t)j * nb] = 0.0;
    }
    return;
  }
  __shared__ double U[TB][TB + 1];  // U[j][i]: entry (i, j), inverted in place
  __shared__ double P[32 * 32];
  for (int e = tid; e < TB * TB; e += 256) {
    const int i = e % TB, j = e / TB;
    U[j][i] = i < j ? (j0 + j < nb ? G[i0 + i + (int64_t)(j0 + j) * nb] : 0.0)
                    : (i == j ? 0.5 : 0.0);
  }
  __syncthreads();
  // the four 16 x 16 diagonal blocks, a lane per column: back substitution
  if (tid < 64) {
    const int base = tid & 48, j = tid & 15;
    double x[16];
#pragma unroll
    for (int i = 15; i >= 0; --i) {
      double sum = 0.0;
#pragma unroll
      for (int k = i + 1; k < 16; ++k) sum += U[base + k][base + i] * x[k];
      x[i] = i == j ? 2.0 : (i < j ? -2.0 * sum : 0.0);
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < 16; ++i) U[base + j][base + i] = x[i];
  }
  __syncthreads();
  for (int s = 16; s < TB; s *= 2) {
    const int tot = TB / 2 * s;  // entries of the TB / (2 s) pairs' B blocks
    for (int e = tid; e < tot; e += 256) {
      const int i = e % s, j = e / s % s, r0 = e / (s * s) * 2 * s;
      double sum = 0.0;
      for (int k = 0; k <= j; ++k) sum += U[r0 + s + k][r0 + i] * U[r0 + s + j][r0 + s + k];
      P[e] = sum;
    }
    __syncthreads();
    for (int e = tid; e < tot; e += 256) {
      const int i = e % s, j = e / s % s, q = e / (s * s), r0 = q * 2 * s;
      double sum = 0.0;
      for (int k = i; k < s; ++k) sum += U[r0 + k][r0 + i] * P[q * s * s + j * s + k];
      U[r0 + s + j][r0 + i] = -sum;
    }
    __syncthreads();
  }
  for (int e = tid; e < TB * TB; e += 256) {
    const int i = e % TB, j = e / TB;
    if (i0 + i < nb && j0 + j < nb) T[i0 + i + (int64_t)(j0 + j) * nb] = U[j][i];
  }
}

// Joins the inverted s x s blocks A (rows r0 = 2 s blockIdx.y) and C (rows
// r0 + s): a group takes 16 columns of the s x s block between them, first
// X = B C^{-1}, kept in LDS, then -A^{-1} X, in 16 x 16 FP64 matrix-core
// blocks over 8 waves (operand layouts: gemm.hip).  s a multiple of 16 up to
// 256; columns from nb on are zeros.
__global__ __launch_bounds__(512) void bt_tmerge(int nb, int s, const double* G, double* T) {
  typedef double d4 __attribute__((ext_vector_type(4)));
  __shared__ double X[256 * 17];
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r0 = 2 * s * blockIdx.y, c0 = blockIdx.x * 16;
  const int rc = r0 + s, col = rc + c0;  // C's first row, this group's first column
  if (col >= nb) return;
  const int kc = c0 + 16;  // rows of C^{-1} above this panel's diagonal
  for (int e = tid; e < kc * 16; e += 512) {
    const int k = e % kc, c = e / kc;
    X[k * 17 + c] = rc + k < nb && col + c < nb ? T[rc + k + (int64_t)(col + c) * nb] : 0.0;
  }
  __syncthreads();
  d4 acc[2] = {d4{0, 0, 0, 0}, d4{0, 0, 0, 0}};
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int t = wave + 8 * q;
    if (16 * t >= s) break;
    const double* g = G + r0 + 16 * t + lr + (int64_t)rc * nb;
#pragma unroll 4
    for (int k = 0; k < kc; k += 4) {
      const double av = rc + k + lq < nb ? g[(int64_t)(k + lq) * nb] : 0.0;
      acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, X[(k + lq) * 17 + lr], acc[q], 0, 0, 0);
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int t = wave + 8 * q;
    if (16 * t >= s) break;
#pragma unroll
    for (int r = 0; r < 4; ++r) X[(16 * t + lq + 4 * r) * 17 + lr] = acc[q][r];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int t = wave + 8 * q;
    if (16 * t >= s) break;
    const double* a = T + r0 + 16 * t + lr + (int64_t)r0 * nb;
    d4 sum = {0, 0, 0, 0};
#pragma unroll 4
    for (int k = 16 * t; k < s; k += 4)
      sum = __builtin_amdgcn_mfma_f64_16x16x4f64(a[(int64_t)(k + lq) * nb],
                                                 X[(k + lq) * 17 + lr], sum, 0, 0, 0);
    if (col + lr < nb) {
      double* o = T + r0 + 16 * t + (int64_t)(col + lr) * nb;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[lq + 4 * r] = -sum[r];
    }
  }
}

int form_t(int nb, const double* G, double* T, hipStream_t st) {
  static_assert(NBB <= 512, "bt_tmerge joins blocks of up to 256");
  const unsigned nt = (unsigned)ceil_div(nb, TB);
  hipLaunchKernelGGL(bt_tdiag, dim3(nt, nt), dim3(256), 0, st, nb, G, T);
  DDC_LAUNCHED();
  for (int s = TB; s < nb; s *= 2) {
    hipLaunchKernelGGL(bt_tmerge, dim3(s / 16, (unsigned)ceil_div(nb, 2 * s)), dim3(512), 0, st,
                       nb, s, G, T);
    DDC_LAUNCHED();
  }
  return DDC_OK;
}

// Library GEMM / triangular solve in the precision of the block.
static int gemm_t(char ta, char tb, int M, int N, int K, double alpha, const double* A, int lda,
                  const double* B, int ldb, double beta, double* C, int ldc, hipStream_t st) {
  return dgemm(ta, tb, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, st);
}
static int gemm_t(char ta, char tb, int M, int N, int K, float alpha, const float* A, int lda,
                  const float* B, int ldb, float beta, float* C, int ldc, hipStream_t st) {
  return sgemm(ta, tb, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, st);
}
static int trsm_t(int M, int N, const double* T, int ldt, double* B, int ldb, hipStream_t st) {
  return dtrsm_left_upper(M, N, T, ldt, B, ldb, st);
}
static int trsm_t(int M, int N, const float* T, int ldt, float* B, int ldb, hipStream_t st) {
  return strsm_left_upper(M, N, T, ldt, B, ldb, st);
}

// The left and right applications are independent: the right one runs on a
// second stream of the device, forked after the unpacking and joined before
// returning, so that the two sequences of block products (each ending in
// small, latency-bound GEMMs and triangular solves) overlap.
struct SideStream {
  hipStream_t s = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
};
constexpr int kMaxSideDev = 64;
static SideStream g_side[kMaxSideDev];

static int side_stream(SideStream** out) {
  int dev = 0;
  DDC_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxSideDev) return DDC_E_ARG;
  SideStream& sd = g_side[dev];
  if (!sd.s) DDC_HIP(hipStreamCreateWithFlags(&sd.s, hipStreamNonBlocking));
  if (!sd.fork) DDC_HIP(hipEventCreateWithFlags(&sd.fork, hipEventDisableTiming));
  if (!sd.join) DDC_HIP(hipEventCreateWithFlags(&sd.join, hipEventDisableTiming));
  *out = &sd;
  return DDC_OK;
}

void backtrans_plan(ArenaPlan& p, int m, int n) {
  p.add<double>((size_t)NBB * NBB * 2);  // G, T
  p.add<double>((size_t)NBB * n);        // Z
  p.add<double>((size_t)m * NBB);        // packed reflectors
  p.add<double>((size_t)NBB * n);        // T Z
  // the right-hand application's own set
  p.add<double>((size_t)NBB * NBB * 2);
  p.add<double>((size_t)NBB * n);
  p.add<double>((size_t)n * NBB);
  p.add<double>((size_t)NBB * n);
}

// Apply H_k0 ... H_k1-1 (blocks, last block first) to the rows of C:
// Z = W^T C, Z = T Z, C -= W Z.  With Z2 (FP64 only): T is formed once per
// block into Ti and applied as a GEMM into Z2 (nb x ncol); else by a triangular
// solve with T^{-1} in place (the solve's blocked small products took about a
// third of the back-transformation at 8192^2).
// left: w_k = A[k:m, k];  right: w_k = A[k, k+1:n] acting on rows k+1..n-1.
template <typename T>
static int apply_blocks(bool left, int m, int n, const T* A, int lda, int nref, T* C, int ldc,
                        int ncol, T* G, T* Ti, T* Z, T* Wd, hipStream_t st, T* Z2 = nullptr) {
  const int nblk = (int)ceil_div(nref, NBB);
  for (int bi = nblk - 1; bi >= 0; --bi) {
    const int k0 = bi * NBB;
    const int nb = std::min(NBB, nref - k0);
    const int rows = left ? m - k0 : n - k0 - 1;
    if (rows <= 0) continue;
    T* Csub = left ? C + k0 : C + k0 + 1;
    dim3 gp((unsigned)ceil_div(rows, 32), (unsigned)ceil_div(nb, 32));
    if (left)
      hipLaunchKernelGGL((bt_pack<false, T>), gp, dim3(32, 8), 0, st, rows, nb,
                         A + k0 + (int64_t)k0 * lda, lda, Wd, rows);
    else
      hipLaunchKernelGGL((bt_pack<true, T>), gp, dim3(32, 8), 0, st, rows, nb,
                         A + k0 + (int64_t)(k0 + 1) * lda, lda, Wd, rows);
    DDC_LAUNCHED();
    DDC_TRY(gemm_t('T', 'N', nb, nb, rows, T(1), Wd, rows, Wd, rows, T(0), G, nb, st));
    DDC_TRY(gemm_t('T', 'N', nb, ncol, rows, T(1), Wd, rows, Csub, ldc, T(0), Z, nb, st));
    T* Zt = Z2 ? Z2 : Z;
    if (Z2) {
      if constexpr (sizeof(T) == 8) {
        DDC_TRY(form_t(nb, G, Ti, st));
        DDC_TRY(gemm_t('N', 'N', nb, ncol, nb, T(1), Ti, nb, Z, nb, T(0), Z2, nb, st));
      }
    } else {
      hipLaunchKernelGGL(bt_tinv<T>, dim3((unsigned)ceil_div(nb * nb, 256)), dim3(256), 0, st, nb,
                         G, Ti);
      DDC_LAUNCHED();
      DDC_TRY(trsm_t(nb, ncol, Ti, nb, Z, nb, st));
    }
    DDC_TRY(gemm_t('N', 'N', rows, ncol, nb, T(-1), Wd, rows, Zt, nb, T(1), Csub, ldc, st));
  }
  return DDC_OK;
}

int backtrans_run(int m, int n, const double* A, int lda, const double* Ut,
                  const double* Vt, int ldb, double* U, int ldu, double* V,
                  int ldv, Arena& ws, hipStream_t st) {
  if (m < n || n < 1) return DDC_E_ARG;
  double* G = ws.take<double>((size_t)NBB * NBB * 2);
  double* Ti = G ? G + NBB * NBB : nullptr;
  double* Z = ws.take<double>((size_t)NBB * n);
  double* Wd = ws.take<double>((size_t)m * NBB);
  double* TZ = ws.take<double>((size_t)NBB * n);
  double* G2 = ws.take<double>((size_t)NBB * NBB * 2);
  double* Ti2 = G2 ? G2 + NBB * NBB : nullptr;
  double* Z2 = ws.take<double>((size_t)NBB * n);
  double* Wd2 = ws.take<double>((size_t)n * NBB);
  double* TZ2 = ws.take<double>((size_t)NBB * n);
  if (!TZ2) return DDC_E_NOMEM;
  SideStream* sd = nullptr;
  DDC_TRY(side_stream(&sd));
  dim3 tb(32, 8);
  dim3 gu((unsigned)ceil_div(n, 32), (unsigned)ceil_div(m, 32));
  hipLaunchKernelGGL(bt_unpack<double>, gu, tb, 0, st, n, m, Ut, ldb, U, ldu);
  DDC_LAUNCHED();
  dim3 gv((unsigned)ceil_div(n, 32), (unsigned)ceil_div(n, 32));
  hipLaunchKernelGGL(bt_unpack<double>, gv, tb, 0, st, n, n, Vt, ldb, V, ldv);
  DDC_LAUNCHED();
  const bool right = n > 2;
  if (right) {
    DDC_HIP(hipEventRecord(sd->fork, st));
    DDC_HIP(hipStreamWaitEvent(sd->s, sd->fork, 0));
  }
  // left: reflectors 0..n-1 (the last one is the 1 x 1 sign flip when m == n)
  const int rcl = apply_blocks(true, m, n, A, lda, n, U, ldu, n, G, Ti, Z, Wd, st, TZ);
  // right: reflectors 0..n-3 (row n-2 holds no reflection); joined even on
  // failure, so that nothing of this call still runs when it returns
  int rcr = DDC_OK;
  if (right) {
    rcr = apply_blocks(false, m, n, A, lda, n - 2, V, ldv, n, G2, Ti2, Z2, Wd2, sd->s, TZ2);
    DDC_HIP(hipEventRecord(sd->join, sd->s));
    DDC_HIP(hipStreamWaitEvent(st, sd->join, 0));
  }
  DDC_TRY(rcl);
  DDC_TRY(rcr);
  return DDC_OK;
}

void backtrans_plan_f32(ArenaPlan& p, int n) {
  for (int side = 0; side < 2; ++side) {
    p.add<float>((size_t)NBB * NBB * 2);
    p.add<float>((size_t)NBB * n);
    p.add<float>((size_t)n * NBB);
  }
}

// FP32 arithmetic throughout (the mixed-precision form refines the result).
int backtrans_run_f32(int n, const float* A32, int lda, const double* Ut, const double* Vt,
                      int ldb, float* U32, float* V32, Arena& ws, hipStream_t st) {
  if (n < 1) return DDC_E_ARG;
  float* G = ws.take<float>((size_t)NBB * NBB * 2);
  float* Ti = G ? G + NBB * NBB : nullptr;
  float* Z = ws.take<float>((size_t)NBB * n);
  float* Wd = ws.take<float>((size_t)n * NBB);
  float* G2 = ws.take<float>((size_t)NBB * NBB * 2);
  float* Ti2 = G2 ? G2 + NBB * NBB : nullptr;
  float* Z2 = ws.take<float>((size_t)NBB * n);
  float* Wd2 = ws.take<float>((size_t)n * NBB);
  if (!Wd2) return DDC_E_NOMEM;
  SideStream* sd = nullptr;
  DDC_TRY(side_stream(&sd));
  dim3 tb(32, 8);
  dim3 g((unsigned)ceil_div(n, 32), (unsigned)ceil_div(n, 32));
  hipLaunchKernelGGL(bt_unpack<float>, g, tb, 0, st, n, n, Ut, ldb, U32, n);
  hipLaunchKernelGGL(bt_unpack<float>, g, tb, 0, st, n, n, Vt, ldb, V32, n);
  DDC_LAUNCHED();
  const bool right = n > 2;
  if (right) {
    DDC_HIP(hipEventRecord(sd->fork, st));
    DDC_HIP(hipStreamWaitEvent(sd->s, sd->fork, 0));
  }
  const int rcl = apply_blocks<float>(true, n, n, A32, lda, n, U32, n, n, G, Ti, Z, Wd, st);
  int rcr = DDC_OK;
  if (right) {
    rcr = apply_blocks<float>(false, n, n, A32, lda, n - 2, V32, n, n, G2, Ti2, Z2, Wd2, sd->s);
    DDC_HIP(hipEventRecord(sd->join, sd->s));
    DDC_HIP(hipStreamWaitEvent(st, sd->join, 0));
  }
  DDC_TRY(rcl);
  DDC_TRY(rcr);
  return DDC_OK;
}

// C (rows x cols, ld ldc) = the leading part of the identity.
__global__ void bt_identity(int rows, int cols, double* C, int ldc) {
  const int64_t total = (int64_t)rows * cols;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t j = e / rows, i = e - j * rows;
    C[i + j * ldc] = i == j ? 1.0 : 0.0;
  }
}

void form_q_plan(ArenaPlan& p, int m, int n, bool left) {
  const int ncol = left ? m : n;
  p.add<double>((size_t)NBB * NBB * 2);
  p.add<double>((size_t)NBB * ncol);
  p.add<double>((size_t)(left ? m : n) * NBB);
}

// Q = H_0 ... H_{n-1} (left, m x m) or G_0 ... G_{n-3} (right, n x n) from the
// reflectors stored in A (m x n, m >= n), as form_u_par / form_v_par build
// them column by column (bidiag_par.c:877-988); here one compact-WY block at
// a time on the identity.
int form_q_run(bool left, int m, int n, const double* A, int lda, double* Q, int ldq, Arena& ws,
               hipStream_t st) {
  if (m < n || n < 1) return DDC_E_ARG;
  const int k = left ? m : n;
  double* G = ws.take<double>((size_t)NBB * NBB * 2);
  double* Ti = G ? G + NBB * NBB : nullptr;
  double* Z = ws.take<double>((size_t)NBB * k);
  double* Wd = ws.take<double>((size_t)k * NBB);
  if (!Wd) return DDC_E_NOMEM;
  const unsigned g = (unsigned)std::min<int64_t>(ceil_div((int64_t)k * k, 256), 8192);
  hipLaunchKernelGGL(bt_identity, dim3(g), dim3(256), 0, st, k, k, Q, ldq);
  DDC_LAUNCHED();
  if (left) return apply_blocks(true, m, n, A, lda, n, Q, ldq, k, G, Ti, Z, Wd, st);
  if (n > 2) return apply_blocks(false, m, n, A, lda, n - 2, Q, ldq, k, G, Ti, Z, Wd, st);
  return DDC_OK;
}

}  // namespace ddc
