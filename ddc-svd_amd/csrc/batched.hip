// batched.hip -- SVD of many small matrices of uneven shapes in one
// persistent launch (FP64 or FP32), replayed from a captured HIP graph.
//
// No reference counterpart: the reference factors one matrix per call
// (svd_gpu.c:53).  Method: one-sided (Hestenes) Jacobi by column blocks,
// one wavefront per matrix.
//
//  * A persistent grid, one workgroup per CU (8 waves in FP64, 12 in FP32 at
//    the default variants: all that the registers allow), pulls matrix
//    indices from an atomic counter; the queue is ordered by descending work
//    (n^2 m), so the large matrices start first and the small ones fill the
//    tail.  A matrix with min(m, n) >= coop_nt is factored by a whole
//    workgroup; from the first smaller matrix on, every wave takes matrices
//    on its own.  Batches of few large matrices last as long as the largest
//    one: 256 x 256 takes 18 ms in FP64 (88 before, with four waves).
//  * A matrix (tall orientation: mt = max(m,n) <= 256 rows, nt = min(m,n)
//    columns; a wide matrix is processed as its transpose) is split into
//    column blocks of width B.  For each block pair (I, J) a wave holds the
//    2B columns of the working matrix and of V in registers (lane l holds rows
//    l, l+64, ...), runs every cross pair (B rounds of B disjoint pairs) and,
//    on the first visit of a block in a sweep, its internal pairs (B-1
//    rounds).  The rounds are unrolled, so that columns stay in their
//    registers; the dot products are summed by lane swaps and DPP.  The
//    squared column norms are reduced once per block pair and then carried
//    through the rotations (alpha' = alpha - t gamma, beta' = beta + t gamma).
//  * In FP32, and for a wave alone, block pairs come from memory and go back.
//    A workgroup takes an FP64 matrix by super-blocks (bj_sweeps_super), one
//    trip to memory for up to 8 x 8 block pairs.
//  * FP32 arithmetic (its order, its roundings, its square roots and
//    divisions) is fixed: vectors of close values show every change of it at
//    the 1e-5 level.
//  * Sweeps stop when every pair satisfies |gamma| <= tol sqrt(alpha beta),
//    tol = sqrt(mt) * eps.  Then sigma_j = ||a_j||, U_j = a_j / sigma_j, and
//    the columns are written in ascending order of sigma.  Columns of exactly
//    zero norm are completed to an orthonormal basis by Gram-Schmidt on unit
//    vectors.
//
// The kernel variant (block width per row class, which also sets the register
// budget and so the waves of a workgroup) decides the order of the rotations
// and with it the last digits of the results: it is picked by the sizes of the
// batch (bj_variant).  The cooperation threshold coop_nt changes no bit, and is
// picked by measurement (svd_gpu_batched_tune).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <numeric>
#include <tuple>
#include <vector>

#include "../../include/svd_gpu.h"
#include "ddc_common.h"
#include "householder.h"

namespace ddc {

constexpr int BJ_MAXDIM = 256;  // max(m, n) of one matrix
constexpr int BJ_MAXSWEEP = 40;

struct BatchItem {
  int m, n;
  int64_t a, s, u, v;  // element offsets of A, sigma, U, V
  int64_t wa, wv;      // element offsets of the working matrix and of V
};

template <typename T>
struct BjArgs {
  int count;
  const BatchItem* items;
  const int* order;  // processing order
  int* counter;      // queue head; zero before the launch
  const T* A;
  T* S;
  T* U;
  T* V;
  T* W;      // working matrices (tall orientation, scaled)
  T* WV;     // working V
  int* info;  // per matrix: sweeps used, or -1 if not converged (may be null)
  int coop_nt;  // matrices with min(m, n) >= coop_nt are factored by a whole workgroup
};

template <typename T>
struct Num;
template <>
struct Num<double> {
  static constexpr double eps = 1.1102230246251565e-16;
  static constexpr double big = 1e150;
};
template <>
struct Num<float> {
  static constexpr float eps = 5.9604645e-08f;
  static constexpr float big = 1e18f;
};

// Raw buffer access to one column of rows entries (rows = 0: a masked column):
// loads past it return 0 and stores there are dropped by the hardware range
// check, so masked rows and columns need no branches, and every column is
// reached from one lane offset (vo, bytes) and a scalar resource.
template <typename T>
struct Col {
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ Col(const T* p, int rows)
      : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(p), 0, rows * (int)sizeof(T),
                                            0x00020000)) {}
  __device__ __forceinline__ T ld(int vo) const;
  __device__ __forceinline__ void st(int vo, T v) const;
};
template <>
__device__ __forceinline__ double Col<double>::ld(int vo) const {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, vo, 0, 0));
}
template <>
__device__ __forceinline__ float Col<float>::ld(int vo) const {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, vo, 0, 0));
}
template <>
__device__ __forceinline__ void Col<double>::st(int vo, double v) const {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(
      decltype(__builtin_amdgcn_raw_buffer_load_b64(r, 0, 0, 0)), v), r, vo, 0, 0);
}
template <>
__device__ __forceinline__ void Col<float>::st(int vo, float v) const {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, vo, 0, 0);
}

// ---- wave sums without LDS: lane swaps and DPP -----------------------------

template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ double dpp_mov(double v) {
  return dpp_all<CTRL>(v);
}
// the value of lane l ^ M (M = 1, 2, 4, 8)
template <int M, typename T>
__device__ __forceinline__ T lane_xor(T v) {
  if constexpr (M == 1) return dpp_mov<DPP_XOR1>(v);
  if constexpr (M == 2) return dpp_mov<DPP_XOR2>(v);
  if constexpr (M == 4) return dpp_mov<DPP_HALF_MIRROR>(dpp_mov<DPP_QUAD_REVERSE>(v));
  if constexpr (M == 8) return dpp_mov<DPP_ROR8>(v);
}
template <int W>
__device__ __forceinline__ void swap_lanes(float& a, float& b) {
  const unsigned x = __float_as_uint(a), y = __float_as_uint(b);
  if constexpr (W == 32) {
    const auto l = __builtin_amdgcn_permlane32_swap(x, y, false, false);
    a = __uint_as_float(l[0]);
    b = __uint_as_float(l[1]);
  } else {
    const auto l = __builtin_amdgcn_permlane16_swap(x, y, false, false);
    a = __uint_as_float(l[0]);
    b = __uint_as_float(l[1]);
  }
}
// v plus the value of lane l ^ W (W = 16, 32)
template <int W, typename T>
__device__ __forceinline__ T add_across(T v) {
  T a = v, b = v;
  swap_lanes<W>(a, b);
  return a + b;
}

// Wave sum of each g[i], delivered to the 64 / N lanes with lane / (64 / N)
// == i, summed across lane bits 5, 4, 3, 2, 1, 0 in this order (as
// reduce_scatter of ddc_common.h, which exchanges through LDS instead).
// lane_scatter_low: the part after lane bit 5 (of the first N / 2 values).
template <typename T, int N>
__device__ __forceinline__ T lane_scatter_low(T (&g)[N]) {
  static_assert(N == 2 || N == 4 || N == 8 || N == 16, "two to sixteen values");
  const int lane = threadIdx.x & 63;
  T v;
  if constexpr (N >= 4) {
#pragma unroll
    for (int j = 0; j < N / 4; ++j) {
      swap_lanes<16>(g[j], g[j + N / 4]);
      g[j] += g[j + N / 4];
    }
  } else {
    g[0] = add_across<16>(g[0]);
  }
  if constexpr (N >= 8) {
    const bool up = (lane >> 3) & 1;
#pragma unroll
    for (int j = 0; j < N / 8; ++j) {
      const T lo = g[j], hi = g[j + N / 8];
      g[j] = (up ? hi : lo) + lane_xor<8>(up ? lo : hi);
    }
  } else {
    g[0] += lane_xor<8>(g[0]);
  }
  if constexpr (N >= 16) {
    const bool up = (lane >> 2) & 1;
    const T lo = g[0], hi = g[1];
    v = (up ? hi : lo) + lane_xor<4>(up ? lo : hi);
  } else {
    v = g[0] + lane_xor<4>(g[0]);
  }
  v += lane_xor<2>(v);
  v += lane_xor<1>(v);
  return v;
}
template <typename T, int N>
__device__ __forceinline__ T lane_scatter(T (&g)[N]) {
#pragma unroll
  for (int j = 0; j < N / 2; ++j) {
    swap_lanes<32>(g[j], g[j + N / 2]);
    g[j] += g[j + N / 2];
  }
  return lane_scatter_low<T, N>(g);
}

template <typename T>
__device__ __forceinline__ T wsum(T v) {
  v = add_across<32>(v);
  v = add_across<16>(v);
  v += lane_xor<8>(v);
  v += lane_xor<4>(v);
  v += lane_xor<2>(v);
  v += lane_xor<1>(v);
  return v;
}

template <typename T>
__device__ __forceinline__ T wmax(T v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return v;
}

// Broadcast of lane l's value (to a wave-uniform register).
__device__ __forceinline__ double rdlane(double x, int l) {
  const long long u = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readlane((int)(u & 0xffffffffll), l);
  const int hi = __builtin_amdgcn_readlane((int)(u >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
__device__ __forceinline__ float rdlane(float x, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

// Jacobi rotation of the pair with squared norms al, be and dot product ga.
// Returns false (no rotation) when the pair is already orthogonal to tol.
template <typename T>
__device__ __forceinline__ bool jrot(T al, T be, T ga, T tol, T& c, T& s, T& t, T& off) {
  const T den = sqrt(al) * sqrt(be);
  if (!(den > T(0)) || !(fabs(ga) > tol * den)) return false;
  off = fmax(off, fabs(ga) / den);
  const T zeta = (be - al) / (T(2) * ga);
  const T az = fabs(zeta);
  const T tm = az > Num<T>::big ? T(0.5) / az : T(1) / (az + sqrt(T(1) + az * az));
  t = zeta < T(0) ? -tm : tm;
  c = T(1) / sqrt(T(1) + t * t);
  s = c * t;
  return true;
}

// In FP64 the square roots and divisions of the general form (about 100
// dependent instructions) are the longest part of a round.  Here the same
// angle comes from half the difference D of the squared norms,
//     t = sign(D) g / (|D| + sqrt(D^2 + g^2)),
// by the hardware's reciprocal and reciprocal square root (about 2^-26) and
// one third-order correction each, to full precision:
//  * D and g are taken relative to the larger norm, so that nothing over- or
//    underflows for columns of any size (a reciprocal of a subnormal dot
//    product is infinite), and the test for orthogonality relative to both;
//    its scales and its bound need the norms alone, which are there before the
//    dot product is.
//  * The dot product that is left is the rounding of the old one.  With a
//    tangent of 26 bits a column in the span of the others loses half as many
//    digits per rotation: 20 to 26 sweeps on constant matrices and on ones of
//    rank 2 and 3, now 11 to 18.
//  * cos^2 + sin^2 must be 1 without bias, as every rotation scales its columns
//    by it: the residual of the cosine's correction is formed from the exact
//    product (two fused multiply-adds).  Over 200 matrices up to 256 x 256 the
//    worst error of a singular value is 5.6e-15 of the largest (6.3e-14 with
//    the tangent of 26 bits and the rounded product, 3.7e-14 with square roots
//    and divisions).
// A batch of 10,000 took 85.4 ms by blocks of 4 (84.9 with the tangent of 26
// bits); it takes 83.8 by the widths of bj_variant.
// off: 1 (the pair was not orthogonal to tol).
template <>
__device__ __forceinline__ bool jrot<double>(double al, double be, double ga, double tol,
                                             double& c, double& s, double& t, double& off) {
  const int ea = __builtin_amdgcn_frexp_exp(al), eb = __builtin_amdgcn_frexp_exp(be);
  const int ex = max(ea, eb), ee = ea + eb;
  const double lim = tol * tol * __builtin_amdgcn_frexp_mant(al) *
                     __builtin_amdgcn_frexp_mant(be) * ((ee & 1) ? 2.0 : 1.0);
  const double D = ldexp(be, -ex - 1) - ldexp(al, -ex - 1);
  const double gr = ldexp(ga, -(ee >> 1));
  // (a zero norm, or a NaN: no rotation)
  if (!(al > 0.0) || !(be > 0.0) || !(gr * gr > lim)) return false;
  off = 1.0;
  const double g = ldexp(ga, -ex);
  const double h = fma(g, g, D * D);
  const double z = __builtin_amdgcn_rsq(h);
  const double p = h * z, e = fma(-p, z, 1.0);
  const double den = fabs(D) + fma(p, e * fma(0.375, e, 0.5), p);
  const double y = __builtin_amdgcn_rcp(den);
  const double f = fma(-den, y, 1.0), t0 = g * y;
  const double tm = fma(t0, fma(f, f, f), t0);
  t = D < 0.0 ? -tm : tm;
  const double q = fma(t, t, 1.0);
  const double x = __builtin_amdgcn_rsq(q);
  const double w = q * x, r = fma(-fma(q, x, -w), x, fma(-w, x, 1.0));
  c = fma(x * r, fma(0.375, r, 0.5), x);
  s = c * t;
  return true;
}

// The 2B columns of a block pair held by one wave: positions 0..B-1 are block
// I, B..2B-1 block J; lane l holds rows l + 64 e.
template <typename T, int B, int R, int RV>
struct Block {
  T a[2 * B][R];
  T v[2 * B][RV];
};

// x y + z.  In FP64 fused wherever it is inlined: left to the compiler, the
// copies of one expression in the sweeps of a workgroup and of a wave alone
// round differently.
template <typename T>
__device__ __forceinline__ T madd(T x, T y, T z) {
  if constexpr (sizeof(T) == 8) return fma(x, y, z);
  else return x * y + z;
}

template <typename T>
__device__ __forceinline__ void turn(T& x, T& y, T c, T s) {
  const T u = x, v = y;
  if constexpr (sizeof(T) == 8) {
    x = fma(c, u, -(s * v));
    y = fma(s, u, c * v);
  } else {
    x = c * u - s * v;
    y = s * u + c * v;
  }
}

template <typename T, int B, int R, int RV>
__device__ __forceinline__ void rotate_cols(Block<T, B, R, RV>& k, int p, int q, T c, T s) {
#pragma unroll
  for (int e = 0; e < R; ++e) turn(k.a[p][e], k.a[q][e], c, s);
#pragma unroll
  for (int e = 0; e < RV; ++e) turn(k.v[p][e], k.v[q][e], c, s);
}

// Cross round S of a block pair: B disjoint rotations, column i of block I
// with column (i + S) mod B of block J.  al, be: the squared norms of the
// lane's group's pair (group i: the 64 / B lanes from 64 / B i).  The dot
// products are scattered over the groups; each group computes its rotation,
// and the cosines and sines are broadcast.  The columns stay where they are
// (S is a constant); only be moves on by one group.
template <typename T, int B, int R, int RV, int S>
__device__ __forceinline__ void cross_round(Block<T, B, R, RV>& k, T& al, T& be, T tol, T& off) {
  constexpr int GS = 64 / B;
  T g[B];
#pragma unroll
  for (int i = 0; i < B; ++i) {
    T d = T(0);
#pragma unroll
    for (int e = 0; e < R; ++e) d = madd(k.a[i][e], k.a[B + (i + S) % B][e], d);
    g[i] = d;
  }
  const T gl = lane_scatter<T, B>(g);
  T c = T(1), s = T(0), t = T(0);
  const bool act = jrot(al, be, gl, tol, c, s, t, off);
  // (the fused forms are spelled out: left to the compiler, a select around
  // them may split the product from the sum)
  const T aln = fmax(__builtin_elementwise_fma(-t, gl, al), T(0));
  const T ben = __builtin_elementwise_fma(t, gl, be);
  al = act ? aln : al;
  be = __shfl(act ? ben : be, ((threadIdx.x & 63) + GS) & 63, 64);
#pragma unroll
  for (int i = 0; i < B; ++i) {
    const T si = rdlane(s, i * GS);
    if (si != T(0)) rotate_cols(k, i, B + (i + S) % B, rdlane(c, i * GS), si);
  }
}
template <typename T, int B, int R, int RV, int S = 0>
__device__ __forceinline__ void cross_rounds(Block<T, B, R, RV>& k, T& al, T& be, T tol, T& off) {
  cross_round<T, B, R, RV, S>(k, al, be, tol, off);
  if constexpr (S + 1 < B) cross_rounds<T, B, R, RV, S + 1>(k, al, be, tol, off);
}

// Internal round S (S < B-1) of both halves: half h's columns meet in pairs by
// the circle method, slot j < B/2 pairing positions j and B-1-j, where
// position 0 holds column 0 and position x > 0 column 1 + (x-1 + S) mod (B-1).
// The columns stay where they are.  nrm: lane c holds the squared norm of
// column c.
template <int B, int S>
__host__ __device__ constexpr int circle(int x) {
  return x == 0 ? 0 : 1 + (x - 1 + S < B - 1 ? x - 1 + S : x - 1 + S - (B - 1));
}
template <typename T, int B, int R, int RV, int S>
__device__ __forceinline__ void intra_round(Block<T, B, R, RV>& k, T& nrm, bool enI, bool enJ,
                                            T tol, T& off) {
  const int lane = threadIdx.x & 63;
  constexpr int GS = 64 / B, H = B / 2;  // lanes per pair, pairs per half
  T g[B];
#pragma unroll
  for (int i = 0; i < B; ++i) {
    T d = T(0);
    if (i < H ? enI : enJ) {
#pragma unroll
      for (int e = 0; e < R; ++e)
        d = madd(k.a[i / H * B + circle<B, S>(i % H)][e],
                 k.a[i / H * B + circle<B, S>(B - 1 - i % H)][e], d);
    }
    g[i] = d;
  }
  const T gl = lane_scatter<T, B>(g);
  const int h = lane / GS / H, j = lane / GS % H;  // the pair this lane's group handles
  const T al = __shfl(nrm, h * B + circle<B, S>(j), 64);
  const T be = __shfl(nrm, h * B + circle<B, S>(B - 1 - j), 64);
  T c = T(1), s = T(0), t = T(0);
  const bool act = jrot(al, be, gl, tol, c, s, t, off);
  const T aln = act ? fmax(__builtin_elementwise_fma(-t, gl, al), T(0)) : al;
  const T ben = act ? __builtin_elementwise_fma(t, gl, be) : be;
  // new norms back to the column lanes: column x is at position pos
  const int x = lane % B, y = x - 1 - S;
  const int pos = x == 0 ? 0 : 1 + (y < 0 ? y + B - 1 : y);
  const bool qside = pos >= H;
  const int slot = lane < 2 * B ? lane / B * H + (qside ? B - 1 - pos : pos) : 0;
  const T np = __shfl(aln, slot * GS, 64), nq = __shfl(ben, slot * GS, 64);
  if (lane < 2 * B) nrm = qside ? nq : np;
#pragma unroll
  for (int i = 0; i < B; ++i) {
    const T si = rdlane(s, i * GS);
    if (si != T(0))
      rotate_cols(k, i / H * B + circle<B, S>(i % H), i / H * B + circle<B, S>(B - 1 - i % H),
                  rdlane(c, i * GS), si);
  }
}
template <typename T, int B, int R, int RV, int S = 0>
__device__ __forceinline__ void intra_rounds(Block<T, B, R, RV>& k, T& nrm, bool enI, bool enJ,
                                             T tol, T& off) {
  intra_round<T, B, R, RV, S>(k, nrm, enI, enJ, tol, off);
  if constexpr (S + 2 < B) intra_rounds<T, B, R, RV, S + 1>(k, nrm, enI, enJ, tol, off);
}

// Half H (0: block I, 1: block J) of a block pair from and to memory: the
// columns from c0 on (c0 < 0, or past nt: masked).
template <int H, typename T, int B, int R, int RV>
__device__ __forceinline__ void load_half(Block<T, B, R, RV>& k, const T* W, const T* WV, int mt,
                                          int nt, int c0) {
  const int vo = (threadIdx.x & 63) * (int)sizeof(T);
  constexpr int STEP = 64 * (int)sizeof(T);
#pragma unroll
  for (int c = 0; c < B; ++c) {
    const bool ok = c0 >= 0 && c0 + c < nt;
    const int cc = ok ? c0 + c : 0;
    const Col<T> ca(W + (int64_t)cc * mt, ok ? mt : 0), cv(WV + (int64_t)cc * nt, ok ? nt : 0);
#pragma unroll
    for (int e = 0; e < R; ++e) k.a[H * B + c][e] = ca.ld(vo + e * STEP);
#pragma unroll
    for (int e = 0; e < RV; ++e) k.v[H * B + c][e] = cv.ld(vo + e * STEP);
  }
}
template <int H, typename T, int B, int R, int RV>
__device__ __forceinline__ void store_half(const Block<T, B, R, RV>& k, T* W, T* WV, int mt, int nt,
                                           int c0) {
  const int vo = (threadIdx.x & 63) * (int)sizeof(T);
  constexpr int STEP = 64 * (int)sizeof(T);
  // the column resources are made anew here instead of being kept through
  // the rounds
  asm volatile("" : "+s"(c0), "+s"(mt), "+s"(nt));
#pragma unroll
  for (int c = 0; c < B; ++c) {
    const bool ok = c0 >= 0 && c0 + c < nt;
    const int cc = ok ? c0 + c : 0;
    const Col<T> ca(W + (int64_t)cc * mt, ok ? mt : 0), cv(WV + (int64_t)cc * nt, ok ? nt : 0);
#pragma unroll
    for (int e = 0; e < R; ++e) ca.st(vo + e * STEP, k.a[H * B + c][e]);
#pragma unroll
    for (int e = 0; e < RV; ++e) cv.st(vo + e * STEP, k.v[H * B + c][e]);
  }
}

// Squared norms of the columns held: column c's on the 32 / B lanes from
// (32 / B) c.
template <typename T, int B, int R, int RV>
__device__ __forceinline__ T col_norms(const Block<T, B, R, RV>& k) {
  T part[2 * B];
  if constexpr (R == 1) {
    // one entry per lane: the squares of lanes l and l + 32 in one fused
    // multiply-add
#pragma unroll
    for (int c = 0; c < B; ++c) {
      T x = k.a[c][0], y = k.a[B + c][0];
      swap_lanes<32>(x, y);
      part[c] = __builtin_elementwise_fma(x, x, y * y);
    }
    return lane_scatter_low<T, 2 * B>(part);
  } else {
#pragma unroll
    for (int c = 0; c < 2 * B; ++c) {
      T s = T(0);
#pragma unroll
      for (int e = 0; e < R; ++e) s = madd(k.a[c][e], k.a[c][e], s);
      part[c] = s;
    }
    return lane_scatter<T, 2 * B>(part);
  }
}

// One block-pair step.  cI / cJ: first columns of the blocks (cJ < 0: block I
// alone).  Returns the largest relative dot product seen by the lane.
template <typename T, int B, int R, int RV>
__device__ __forceinline__ T block_step(T* __restrict__ W, T* __restrict__ WV, int mt, int nt,
                                        int cI, int cJ, bool intraI, bool intraJ, T tol) {
  const int lane = threadIdx.x & 63;
  cI = __builtin_amdgcn_readfirstlane(cI);
  cJ = __builtin_amdgcn_readfirstlane(cJ);
  Block<T, B, R, RV> k;
  load_half<0>(k, W, WV, mt, nt, cI);
  load_half<1>(k, W, WV, mt, nt, cJ);
  constexpr int GN = 32 / B, GS = 64 / B;  // lanes per column, per pair
  T nrm = col_norms(k);
  T off = T(0);
  T al, be;
  if (intraI || intraJ) {
    nrm = __shfl(nrm, (lane & (2 * B - 1)) * GN, 64);
    intra_rounds(k, nrm, intraI, intraJ, tol, off);
    al = __shfl(nrm, lane / GS, 64);
    be = __shfl(nrm, B + lane / GS, 64);
  } else {
    al = __shfl(nrm, lane / GS * GN, 64);
    be = __shfl(nrm, (B + lane / GS) * GN, 64);
  }
  if (cJ >= 0) cross_rounds(k, al, be, tol, off);
  store_half<0>(k, W, WV, mt, nt, cI);
  store_half<1>(k, W, WV, mt, nt, cJ);
  return off;
}

// Pair i of round r of the round-robin schedule of P players (circle method):
// every pair of 0..P-1 (P even) appears once in rounds 0..P-2.
// (r < P - 1 and i < P / 2: the remainder by P - 1 is one subtraction)
__host__ __device__ constexpr int rr_mod(int P, int x) { return x >= P - 1 ? x - (P - 1) : x; }
__host__ __device__ constexpr int rr_p(int P, int r, int i) {
  return i == 0 ? 0 : 1 + rr_mod(P, i - 1 + r);
}
__host__ __device__ constexpr int rr_q(int P, int r, int i) {
  return 1 + rr_mod(P, P - 2 - i + r);
}

// A team: the nw waves of a workgroup that factor one matrix together
// (nw = 1: a wave alone).  w is the wave's index in the team.
struct Team {
  int w, nw;
  __device__ __forceinline__ void sync() const {
    if (nw > 1) {
      __syncthreads();
    } else {
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }
};

template <typename T>
__device__ __forceinline__ T team_max(T v, Team t, T* red) {
  v = wmax(v);
  if (t.nw == 1) return v;
  if ((threadIdx.x & 63) == 0) red[t.w] = v;
  __syncthreads();
  T r = red[0];
  for (int i = 1; i < t.nw; ++i) r = fmax(r, red[i]);
  __syncthreads();
  return r;
}

// Sweeps of one matrix; returns the sweeps used or -1.  Each sweep is nbe-1
// rounds of the round-robin ordering of the nbe (nb rounded up to even)
// column blocks: the nbe/2 block pairs of a round are disjoint, so the
// team's waves take them in turn.  Round 0 also runs every block's internal
// pairs; a block paired with the dummy block nb runs alone.
template <typename T, int B, int R, int RV>
__device__ __forceinline__ int bj_sweeps(T* W, T* WV, int mt, int nt, Team t, T* red) {
  const T tol = Num<T>::eps * sqrt(T(mt));
  mt = __builtin_amdgcn_readfirstlane(mt);
  nt = __builtin_amdgcn_readfirstlane(nt);
  const int nb = (nt + B - 1) / B;
  const int nbe = nb + (nb & 1);
  const int w = __builtin_amdgcn_readfirstlane(t.w), nw = __builtin_amdgcn_readfirstlane(t.nw);
  for (int sw = 0; sw < BJ_MAXSWEEP; ++sw) {
    T off = T(0);
    for (int r = 0; r < nbe - 1; ++r) {
      for (int i = w; i < nbe / 2; i += nw) {
        int I = rr_p(nbe, r, i), J = rr_q(nbe, r, i);
        if (I > J) {
          const int x = I;
          I = J;
          J = x;
        }
        const bool alone = J >= nb;
        if (alone && r != 0) continue;
        off = fmax(off, block_step<T, B, R, RV>(W, WV, mt, nt, I * B, alone ? -1 : J * B, r == 0,
                                                r == 0 && !alone, tol));
      }
      t.sync();
    }
    off = team_max(off, t, red);
    if (!(off > tol)) return sw + 1;
  }
  return -1;
}

// The sweeps of one FP64 matrix by a whole workgroup (nw waves).  Taking each
// block pair from memory and back, as above, moves the matrix and V through
// L2 and the Infinity Cache once per round: 16 B (m + n) per rotation and
// column pair at B = 4, 3.9 TB/s over a batch of 10,000, and each round waits
// for it.  Here the column blocks are grouped by q <= nw into super-blocks.
//  * Pairs inside the super-blocks: as above, all super-blocks side by side.
//  * Pairs across super-blocks S < T: wave w holds block w of S in registers
//    while every T passes by; block w of T, then its successors, come from
//    the neighbouring wave through LDS, so all q x q pairs are met with one
//    trip to memory for T (and one per S for all T).
// xch: 64 B (R + RV) values per wave.
template <typename T, int B, int R, int RV>
__device__ __forceinline__ int bj_sweeps_super(T* W, T* WV, int mt, int nt, Team t, T* red,
                                               T* xch) {
  const T tol = Num<T>::eps * sqrt(T(mt));
  const int lane = threadIdx.x & 63;
  mt = __builtin_amdgcn_readfirstlane(mt);
  nt = __builtin_amdgcn_readfirstlane(nt);
  const int w = __builtin_amdgcn_readfirstlane(t.w), nw = __builtin_amdgcn_readfirstlane(t.nw);
  const int nb = (nt + B - 1) / B;
  const int ns = (nb + nw - 1) / nw, q = (nb + ns - 1) / ns;
  const int qe = q + (q & 1), hq = qe / 2;
  constexpr int HW = B * (R + RV) * 64;  // values of half a block pair
  constexpr int GN = 32 / B, GS = 64 / B;
  const int next = w + 1 < q ? w + 1 : 0;
  for (int sw = 0; sw < BJ_MAXSWEEP; ++sw) {
    T off = T(0);
    for (int r = 0; r < max(qe - 1, 1); ++r) {
      for (int i = w; i < ns * hq; i += nw) {
        const int s = i / hq, pi = i - s * hq;
        const int x = rr_p(qe, r, pi), y = rr_q(qe, r, pi);
        const int lo = min(x, y), hi = max(x, y);
        const int I = s * q + lo, J = s * q + hi;
        const bool alone = hi >= q || J >= nb;
        if (I >= nb || (alone && r != 0)) continue;
        off = fmax(off, block_step<T, B, R, RV>(W, WV, mt, nt, I * B, alone ? -1 : J * B, r == 0,
                                                r == 0 && !alone, tol));
      }
      t.sync();
    }
    // (waves past q go along with masked columns: branches around parts of
    // the loops would cost the others copies of all their columns)
    for (int S = 0; S + 1 < ns; ++S) {
      Block<T, B, R, RV> k;
      load_half<0>(k, W, WV, mt, nt, w < q ? (S * q + w) * B : -1);
      for (int U = S + 1; U < ns; ++U) {
        load_half<1>(k, W, WV, mt, nt, w < q ? (U * q + w) * B : -1);
#pragma unroll 1
        for (int r = 0;;) {
          const T nrm = col_norms(k);
          T al = __shfl(nrm, lane / GS * GN, 64), be = __shfl(nrm, (B + lane / GS) * GN, 64);
          cross_rounds(k, al, be, tol, off);
          if (++r == q) break;
#pragma unroll
          for (int c = 0; c < B; ++c) {
            T* to = xch + w * HW + c * (R + RV) * 64 + lane;
#pragma unroll
            for (int e = 0; e < R; ++e) to[e * 64] = k.a[B + c][e];
#pragma unroll
            for (int e = 0; e < RV; ++e) to[(R + e) * 64] = k.v[B + c][e];
          }
          __syncthreads();
#pragma unroll
          for (int c = 0; c < B; ++c) {
            const T* from = xch + next * HW + c * (R + RV) * 64 + lane;
#pragma unroll
            for (int e = 0; e < R; ++e) k.a[B + c][e] = from[e * 64];
#pragma unroll
            for (int e = 0; e < RV; ++e) k.v[B + c][e] = from[(R + e) * 64];
          }
          __syncthreads();
        }
        // block w + q - 1 (mod q) of U is here now
        store_half<1>(k, W, WV, mt, nt, w < q ? (U * q + (w > 0 ? w - 1 : q - 1)) * B : -1);
        t.sync();
      }
      store_half<0>(k, W, WV, mt, nt, w < q ? (S * q + w) * B : -1);
      t.sync();
    }
    off = team_max(off, t, red);
    if (!(off > tol)) return sw + 1;
  }
  return -1;
}

// The same sweeps by a wave alone, one block pair after another.  The pairs of
// a round are disjoint, so every column sees the same rotations in the same
// order as with NW waves: which matrices a workgroup takes together is a
// question of time alone, and the results are the same bit for bit.
template <typename T, int B, int R, int RV, int NW>
__device__ __forceinline__ int bj_sweeps_alone(T* W, T* WV, int mt, int nt, Team t) {
  const T tol = Num<T>::eps * sqrt(T(mt));
  mt = __builtin_amdgcn_readfirstlane(mt);
  nt = __builtin_amdgcn_readfirstlane(nt);
  const int nb = (nt + B - 1) / B;
  const int ns = (nb + NW - 1) / NW, q = (nb + ns - 1) / ns;
  const int qe = q + (q & 1), hq = qe / 2;
  const int inside = max(qe - 1, 1);  // rounds inside the super-blocks
  for (int sw = 0; sw < BJ_MAXSWEEP; ++sw) {
    T off = T(0);
    int S = 0, U = 1, d = 0;  // across: block w of S with block w + d of U
    for (int r = 0; r < inside || S + 1 < ns; ++r) {
      const bool in = r < inside;
      for (int i = 0; i < (in ? ns * hq : q); ++i) {
        int I = S * q + i, J = U * q + (i + d < q ? i + d : i + d - q);
        bool alone = false;
        if (in) {
          const int s = i / hq, pi = i - s * hq;
          const int x = rr_p(qe, r, pi), y = rr_q(qe, r, pi);
          I = s * q + min(x, y);
          J = s * q + max(x, y);
          alone = max(x, y) >= q || J >= nb;
        }
        if (I >= nb || (J >= nb && !alone) || (alone && r != 0)) continue;
        off = fmax(off, block_step<T, B, R, RV>(W, WV, mt, nt, I * B, alone ? -1 : J * B, r == 0,
                                                r == 0 && !alone, tol));
      }
      t.sync();
      if (!in && ++d == q) {
        d = 0;
        if (++U == ns) U = ++S + 1;
      }
    }
    if (!(wmax(off) > tol)) return sw + 1;
  }
  return -1;
}

// Copies A (transposed when wide) into W scaled by a power of two so that
// max |a| is in [0.5, 1), and sets WV = I.  Returns the scale.
template <typename T>
__device__ T bj_load(const BatchItem& it, const T* A, T* W, T* WV, int mt, int nt, Team t,
                     T* red) {
  const int lane = threadIdx.x & 63;
  const bool wide = it.m < it.n;
  const T* src = A + it.a;
  T amax = T(0);
  for (int j = t.w; j < nt; j += t.nw)
    for (int r = lane; r < mt; r += 64) {
      const T x = wide ? src[j + (int64_t)r * it.m] : src[r + (int64_t)j * it.m];
      amax = fmax(amax, fabs(x));
    }
  amax = team_max(amax, t, red);
  T scale = T(1);
  if (amax > T(0) && isfinite(amax)) {
    int ex;
    (void)frexp(amax, &ex);
    scale = ldexp(T(1), -ex);
  }
  for (int j = t.w; j < nt; j += t.nw) {
    for (int r = lane; r < mt; r += 64) {
      const T x = wide ? src[j + (int64_t)r * it.m] : src[r + (int64_t)j * it.m];
      W[r + (int64_t)j * mt] = x * scale;
    }
    for (int r = lane; r < nt; r += 64) WV[r + (int64_t)j * nt] = r == j ? T(1) : T(0);
  }
  t.sync();
  return scale;
}

// sigma, ranks (ascending), outputs in order, completion of zero columns.
template <typename T>
__device__ void bj_finish(const BatchItem& it, const BjArgs<T>& g, T* W, T* WV, int mt, int nt,
                          T scale, T* sig, int* rk, Team t) {
  const int lane = threadIdx.x & 63;
  const int tt = t.w * 64 + lane;
  const bool wide = it.m < it.n;
  for (int j = t.w; j < nt; j += t.nw) {
    T s = T(0);
    for (int r = lane; r < mt; r += 64) {
      const T x = W[r + (int64_t)j * mt];
      s += x * x;
    }
    s = wsum(s);
    if (lane == 0) sig[j] = sqrt(s);
  }
  t.sync();
  for (int j = tt; j < nt; j += 64 * t.nw) {
    const T sj = sig[j];
    int c = 0;
    for (int i = 0; i < nt; ++i) {
      const T si = sig[i];
      c += (si < sj || (si == sj && i < j)) ? 1 : 0;
    }
    rk[j] = c;
  }
  int nzero = 0;
  for (int i = 0; i < nt; ++i) nzero += sig[i] == T(0) ? 1 : 0;
  t.sync();
  // Y receives the normalised working columns (mt rows), Z the columns of V (nt rows)
  T* Y = wide ? g.V + it.v : g.U + it.u;
  T* Z = wide ? g.U + it.u : g.V + it.v;
  for (int j = t.w; j < nt; j += t.nw) {
    const int rj = rk[j];
    const T sj = sig[j];
    const T inv = sj > T(0) ? T(1) / sj : T(0);
    for (int r = lane; r < mt; r += 64) Y[r + (int64_t)rj * mt] = W[r + (int64_t)j * mt] * inv;
    for (int r = lane; r < nt; r += 64) Z[r + (int64_t)rj * nt] = WV[r + (int64_t)j * nt];
    if (lane == 0) g.S[it.s + rj] = sj / scale;
  }
  t.sync();
  // zero singular values sort first: columns 0..nzero-1 of Y are zero
  if (t.w == 0) {
    for (int z = 0; z < nzero; ++z) {
      for (int cand = 0; cand < mt; ++cand) {
        T x[BJ_MAXDIM / 64];
#pragma unroll
        for (int e = 0; e < BJ_MAXDIM / 64; ++e) x[e] = (lane + 64 * e == cand) ? T(1) : T(0);
        for (int pass = 0; pass < 2; ++pass) {
          for (int c = 0; c < nt; ++c) {
            if (c >= z && c < nzero) continue;
            T d = T(0);
#pragma unroll
            for (int e = 0; e < BJ_MAXDIM / 64; ++e) {
              const int r = lane + 64 * e;
              if (r < mt) d += Y[r + (int64_t)c * mt] * x[e];
            }
            d = wsum(d);
#pragma unroll
            for (int e = 0; e < BJ_MAXDIM / 64; ++e) {
              const int r = lane + 64 * e;
              if (r < mt) x[e] -= d * Y[r + (int64_t)c * mt];
            }
          }
        }
        T n2 = T(0);
#pragma unroll
        for (int e = 0; e < BJ_MAXDIM / 64; ++e) n2 += x[e] * x[e];
        n2 = wsum(n2);
        if (n2 > T(0.25)) {
          const T inv = T(1) / sqrt(n2);
#pragma unroll
          for (int e = 0; e < BJ_MAXDIM / 64; ++e) {
            const int r = lane + 64 * e;
            if (r < mt) Y[r + (int64_t)z * mt] = x[e] * inv;
          }
          break;
        }
      }
    }
  }
  t.sync();
}

__device__ __forceinline__ int64_t uni64(int64_t x) {
  const int lo = __builtin_amdgcn_readfirstlane((int)(x & 0xffffffffll));
  const int hi = __builtin_amdgcn_readfirstlane((int)(x >> 32));
  return ((int64_t)hi << 32) | (int64_t)(unsigned)lo;
}

template <typename T, int B, int R, int RV, int NW>
__device__ __forceinline__ void bj_matrix(const BatchItem& it, const BjArgs<T>& g, int k,
                                          Team t, T* sig, int* rk, T* red, T* xch) {
  const int mt = it.m > it.n ? it.m : it.n, nt = it.m > it.n ? it.n : it.m;
  T* W = (T*)uni64((int64_t)(g.W + it.wa));
  T* WV = (T*)uni64((int64_t)(g.WV + it.wv));
  const T scale = bj_load(it, g.A, W, WV, mt, nt, t, red);
  int sweeps;
  if constexpr (sizeof(T) == 8)
    sweeps = t.nw > 1 ? bj_sweeps_super<T, B, R, RV>(W, WV, mt, nt, t, red, xch)
                      : bj_sweeps_alone<T, B, R, RV, NW>(W, WV, mt, nt, t);
  else
    sweeps = bj_sweeps<T, B, R, RV>(W, WV, mt, nt, t, red);
  bj_finish(it, g, W, WV, mt, nt, scale, sig, rk, t);
  if (g.info && threadIdx.x % (64 * t.nw) == 0) g.info[k] = sweeps;
}

// The descriptor as wave-uniform (scalar) values.
__device__ __forceinline__ BatchItem uniform_item(const BatchItem& x) {
  BatchItem y;
  y.m = __builtin_amdgcn_readfirstlane(x.m);
  y.n = __builtin_amdgcn_readfirstlane(x.n);
  y.a = uni64(x.a);
  y.s = uni64(x.s);
  y.u = uni64(x.u);
  y.v = uni64(x.v);
  y.wa = uni64(x.wa);
  y.wv = uni64(x.wv);
  return y;
}

__device__ __forceinline__ int pop_wave(int* counter) {
  int idx = 0;
  if ((threadIdx.x & 63) == 0) idx = atomicAdd(counter, 1);
  return __builtin_amdgcn_readfirstlane(idx);
}

// Persistent kernel, one workgroup per CU.  While the queue head holds
// matrices with min(m, n) >= coop_nt, the workgroup's waves factor each one
// together; from the first smaller matrix on (the queue is sorted by work)
// every wave takes matrices on its own.
// B12 / B34: block width for matrices with up to 128 / up to 256 rows.
// MINW: resident waves per SIMD the register allocation must allow.
template <typename T, int B12, int B34, int MINW>
__global__ __launch_bounds__(256 * MINW, MINW) void bj_kernel(BjArgs<T> g) {
  constexpr int WGW = 4 * MINW;  // waves per workgroup: all that a CU holds
  __shared__ T sig[WGW][BJ_MAXDIM];
  __shared__ int rk[WGW][BJ_MAXDIM];
  __shared__ T red[WGW];
  // bj_sweeps_super: at most 2 + 2 values per lane and column up to 128 rows,
  // 4 + 4 beyond
  constexpr int XW = sizeof(T) == 8 ? 64 * (B12 * 4 > B34 * 8 ? B12 * 4 : B34 * 8) : 1;
  __shared__ T xch[WGW * XW];
  __shared__ int s_idx;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  Team t{w, WGW};
  bool coop = true;
  for (;;) {
    int idx;
    if (coop) {
      if (threadIdx.x == 0) s_idx = atomicAdd(g.counter, 1);
      __syncthreads();
      idx = __builtin_amdgcn_readfirstlane(s_idx);
      __syncthreads();
    } else {
      idx = pop_wave(g.counter);
    }
    if (idx >= g.count) return;
    int k = __builtin_amdgcn_readfirstlane(g.order[idx]);
    BatchItem it = uniform_item(g.items[k]);
    if (coop && (it.m < it.n ? it.m : it.n) < g.coop_nt) {
      coop = false;
      t = Team{0, 1};
      if (w != 0) {  // wave 0 keeps this matrix, the others draw their own
        idx = pop_wave(g.counter);
        if (idx >= g.count) return;
        k = __builtin_amdgcn_readfirstlane(g.order[idx]);
        it = uniform_item(g.items[k]);
      }
    }
    T* sg = sig[coop ? 0 : w];
    int* rkk = rk[coop ? 0 : w];
    T* rd = coop ? red : red + w;
    const int mt = it.m > it.n ? it.m : it.n, nt = it.m > it.n ? it.n : it.m;
    const int R = (mt + 63) / 64, RV = (nt + 63) / 64;
#define BJ_CASE(R_, RV_)                                                  \
  if (R == R_ && RV == RV_) {                                             \
    bj_matrix<T, (R_ <= 2 ? B12 : B34), R_, RV_, WGW>(it, g, k, t, sg, rkk, rd, xch); \
    continue;                                                             \
  }
    BJ_CASE(1, 1)
    BJ_CASE(2, 1)
    BJ_CASE(2, 2)
    BJ_CASE(3, 1)
    BJ_CASE(3, 2)
    BJ_CASE(3, 3)
    BJ_CASE(4, 1)
    BJ_CASE(4, 2)
    BJ_CASE(4, 3)
    BJ_CASE(4, 4)
#undef BJ_CASE
  }
}

__global__ void k_fill_i32(int* p, int v, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

struct BjVariant {
  int b12, b34;
  int w64, w32;  // waves per SIMD
  const void* f64;
  const void* f32;
};

#define BJ_VARIANT(B12, B34, W64, W32) \
  {B12, B34, W64, W32, (const void*)&bj_kernel<double, B12, B34, W64>, \
   (const void*)&bj_kernel<float, B12, B34, W32>}
static const BjVariant kVariants[] = {
    BJ_VARIANT(8, 4, 2, 3),
    BJ_VARIANT(4, 4, 2, 3),
    BJ_VARIANT(4, 2, 3, 4),
    BJ_VARIANT(2, 2, 3, 4),
};
#undef BJ_VARIANT
constexpr int kNumVariants = sizeof(kVariants) / sizeof(kVariants[0]);
// thresholds that the tuner times, the first one and those below it, then those
// above it in rising order
static const int kCoopNt[] = {32, 1, 8, 12, 16, 20, 24, 40, 48, 64, 96, 128, BJ_MAXDIM + 1};

// A launch configuration: kernel variant, resident workgroups per CU, and
// the smallest min(m, n) a whole workgroup factors together.
struct BjConfig {
  int variant = -1, wgs = 0, coop_nt = 0;
};

template <typename T>
static int bj_launch(const BjConfig& c, int cus, BjArgs<T> a, hipStream_t st) {
  const BjVariant& v = kVariants[c.variant];
  const void* f = sizeof(T) == 8 ? v.f64 : v.f32;
  a.coop_nt = c.coop_nt;
  const int threads = 256 * (sizeof(T) == 8 ? v.w64 : v.w32);
  void* params[] = {&a};
  DDC_HIP(hipLaunchKernel(f, dim3(cus * c.wgs), dim3(threads), params, 0, st));
  return DDC_OK;
}

// tuned thresholds by (dtype, variant, log2 count, log2 work)
static std::mutex g_tune_mu;
static std::map<std::tuple<int, int, int, int>, int> g_tune_cache;

}  // namespace ddc

struct svd_gpu_batch {
  int count = 0, dtype = 0, cus = 0, dev = 0;
  std::vector<int> m, n;
  std::vector<long long> offA, offS, offU, offV;
  std::vector<int> order;
  double work = 0.0;
  ddc::BatchItem* d_items = nullptr;
  int* d_order = nullptr;   // processing order
  int* d_counter = nullptr;  // [0] queue head
  void* d_work = nullptr;
  size_t work_elems_a = 0, work_elems_v = 0;
  ddc::BjConfig cfg;
  hipStream_t cap = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  const void* gA = nullptr;
  void *gS = nullptr, *gU = nullptr, *gV = nullptr;
  int* ginfo = nullptr;
  std::mutex mu;
};

namespace ddc {

template <typename T>
static BjArgs<T> bj_args(svd_gpu_batch* p, const void* dA, void* dS, void* dU, void* dV,
                         int* info) {
  BjArgs<T> a;
  a.count = p->count;
  a.items = p->d_items;
  a.order = p->d_order;
  a.counter = p->d_counter;
  a.A = (const T*)dA;
  a.S = (T*)dS;
  a.U = (T*)dU;
  a.V = (T*)dV;
  a.W = (T*)p->d_work;
  a.WV = (T*)p->d_work + p->work_elems_a;
  a.info = info;
  return a;
}

static int bj_enqueue(svd_gpu_batch* p, const BjConfig& c, const void* dA, void* dS, void* dU,
                      void* dV, int* info, hipStream_t st) {
  int* ctr = p->d_counter;
  hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(64), 0, st, ctr, 0, 1);
  DDC_LAUNCHED();
  if (p->dtype == SVD_GPU_F64)
    return bj_launch<double>(c, p->cus, bj_args<double>(p, dA, dS, dU, dV, info), st);
  return bj_launch<float>(c, p->cus, bj_args<float>(p, dA, dS, dU, dV, info), st);
}

// Milliseconds of one launch of configuration c on the whole batch (best of 2;
// one alone where it is far from best, the time to beat).
static int bj_time(svd_gpu_batch* p, const BjConfig& c, const void* dA, void* dS, void* dU,
                   void* dV, hipStream_t st, hipEvent_t e0, hipEvent_t e1, float best, float& ms) {
  ms = 1e30f;
  for (int rep = 0; rep < 2 && !(rep > 0 && ms > 1.2f * best); ++rep) {
    DDC_HIP(hipEventRecord(e0, st));
    DDC_TRY(bj_enqueue(p, c, dA, dS, dU, dV, nullptr, st));
    DDC_HIP(hipEventRecord(e1, st));
    DDC_HIP(hipEventSynchronize(e1));
    float t = 0.f;
    DDC_HIP(hipEventElapsedTime(&t, e0, e1));
    ms = std::min(ms, t);
  }
  return DDC_OK;
}

// The variant of a batch, 0 (blocks of 8 up to 128 rows, of 4 beyond) or 1
// (blocks of 4), by its sizes: a timing would pick one or the other from run to
// run where they are close, and the results differ in their last digits (in
// vectors of close values by more).  The narrower ones have more waves at work
// on a matrix, the wider ones pass over it half as often.  ms, 8 | 4 wide, each
// at its best threshold:
//  * FP64, load = work / (CUs x work of the largest):
//      up to 40 columns, few matrices: 24 x 24, 256 of them, 0.29 | 0.18, 512
//      0.50 | 0.33, 1024 0.52 | 0.64; 800 up to 40 x 40 (load 0.43) 0.47 | 0.39,
//      1600 (0.86) 0.61 | 0.67;
//      up to 8 columns, which one block of 8 leaves no other: 2048 of 8 x 8
//      0.13 | 0.10, 3000 of 128 x 8 0.21 | 0.16;
//      more columns: 200 of 128 x 128 2.7 | 3.5, 2000 20 | 26, 10,000 up to 128
//      15.5 | 17.4, up to 256 84.3 | 85.3, 300 up to 64 0.60 | 0.61; the other
//      way by at most a tenth (1600 up to 96 2.63 | 2.41, 800 up to 64
//      0.70 | 0.65);
//      all of more than 128 rows: one width and one result, 0 to 5% in favour of
//      the kernel that holds it alone (8000 of 200 x 8 0.482 | 0.458).
//  * FP32: blocks of 8 wherever the matrices of up to 128 rows and more than 8
//    columns count (10,000 up to 128 13.3 | 15.7, 2000 of 128 x 128 16.6 | 22.2;
//    1536 of 24 x 24 0.58 | 0.77, but 512 0.54 | 0.35); up to 8 columns of 4 (2000
//    of 8 x 8 0.149 | 0.114, one 0.082 | 0.056, 2000 of 200 x 8 0.155 | 0.140).
//    Where one of more than 224 rows outlasts the others the two are within 1%
//    (150 up to 256 12.1 | 12.0, 600 12.7 | 12.8, 2,500 19.6 | 19.5), so the line
//    between them costs nothing wherever it lies.
static int bj_variant(const svd_gpu_batch* p) {
  int rows = 0, least = BJ_MAXDIM, cols = 0;
  double most = 0.0;
  for (int k = 0; k < p->count; ++k) {
    const int mt = std::max(p->m[k], p->n[k]), nt = std::min(p->m[k], p->n[k]);
    rows = std::max(rows, mt);
    least = std::min(least, mt);
    cols = std::max(cols, nt);
    most = std::max(most, (double)nt * nt * mt);
  }
  if (p->dtype == SVD_GPU_F32)
    return cols <= 8 || (rows > 224 && p->work < 350.0 * most) ? 1 : 0;
  const bool few = p->count <= 2 * p->cus || p->work < 0.6 * p->cus * most;
  return cols <= 8 || least > 128 || (cols <= 40 && few) ? 1 : 0;
}

static std::tuple<int, int, int, int> tune_key(const svd_gpu_batch* p) {
  return {p->dtype, bj_variant(p), (int)std::lround(std::log2((double)p->count)),
          (int)std::lround(std::log2(p->work + 1.0))};
}

// The autotuner: times the thresholds, each on the whole batch, but those that
// split it as an earlier one does and, once a larger one takes twice the best
// time, the ones beyond.  (A half-size sample was tried: it keeps the largest
// matrices, whose latency floors the makespan, but only half of the bulk,
// and ranked configurations 25% apart in the wrong order.)
static int bj_tune(svd_gpu_batch* p, const void* dA, void* dS, void* dU, void* dV,
                   hipStream_t st) {
  hipEvent_t e0, e1;
  DDC_HIP(hipEventCreate(&e0));
  if (hipEventCreate(&e1) != hipSuccess) {
    (void)hipEventDestroy(e0);
    return DDC_E_HIP;
  }
  float best = 1e30f;
  BjConfig bc, c;
  c.variant = bj_variant(p);
  c.wgs = 1;  // one workgroup holds all the waves a CU can
  int rc = DDC_OK;
  int seen[sizeof(kCoopNt) / sizeof(kCoopNt[0])], ns = 0;  // matrices taken by whole workgroups
  for (int ct : kCoopNt) {
    int whole = 0;
    for (int k = 0; k < p->count; ++k) whole += std::min(p->m[k], p->n[k]) >= ct;
    if (std::find(seen, seen + ns, whole) != seen + ns) continue;
    seen[ns++] = whole;
    c.coop_nt = ct;
    float ms;
    if ((rc = bj_time(p, c, dA, dS, dU, dV, st, e0, e1, best, ms))) break;
    if (ms < best) {
      best = ms;
      bc = c;
    } else if (ct > kCoopNt[0] && ms > 2.0f * best) {
      break;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (rc) return rc;
  p->cfg = bc;
  std::lock_guard<std::mutex> lk(g_tune_mu);
  g_tune_cache[tune_key(p)] = bc.coop_nt;
  return DDC_OK;
}

static void bj_free(svd_gpu_batch* p) {
  if (p->exec) (void)hipGraphExecDestroy(p->exec);
  if (p->graph) (void)hipGraphDestroy(p->graph);
  if (p->cap) (void)hipStreamDestroy(p->cap);
  if (p->d_items) (void)hipFree(p->d_items);
  if (p->d_order) (void)hipFree(p->d_order);
  if (p->d_counter) (void)hipFree(p->d_counter);
  if (p->d_work) (void)hipFree(p->d_work);
  p->exec = nullptr;
  p->graph = nullptr;
  p->cap = nullptr;
  p->d_items = nullptr;
  p->d_order = nullptr;
  p->d_counter = nullptr;
  p->d_work = nullptr;
}

// Items (element offsets into the packed buffers and into the work area)
// and costs of a batch, in batch order; off* (count + 1 entries) may be
// null.  wa / wv: elements of the working copies of A and V.
static void bj_layout(int count, const int* m, const int* n, BatchItem* items, double* cost,
                      long long* offA, long long* offS, long long* offU, long long* offV,
                      int64_t& wa, int64_t& wv) {
  long long oa = 0, os = 0, ou = 0, ov = 0;
  wa = wv = 0;
  for (int k = 0; k < count; ++k) {
    const int mk = m[k], nk = n[k], mn = std::min(mk, nk), mt = std::max(mk, nk);
    if (offA) {
      offA[k] = oa;
      offS[k] = os;
      offU[k] = ou;
      offV[k] = ov;
    }
    BatchItem& it = items[k];
    it.m = mk;
    it.n = nk;
    it.a = oa;
    it.s = os;
    it.u = ou;
    it.v = ov;
    it.wa = wa;
    it.wv = wv;
    oa += (long long)mk * nk;
    os += mn;
    ou += (long long)mk * mn;
    ov += (long long)nk * mn;
    wa += (int64_t)mt * mn;
    wv += (int64_t)mn * mn;
    cost[k] = (double)mn * mn * mt;
  }
  if (offA) {
    offA[count] = oa;
    offS[count] = os;
    offU[count] = ou;
    offV[count] = ov;
  }
}

static int bj_plan(svd_gpu_batch* p, int count, const int* m, const int* n, int dtype) {
  const size_t es = dtype == SVD_GPU_F64 ? 8 : 4;
  p->count = count;
  p->dtype = dtype;
  p->m.assign(m, m + count);
  p->n.assign(n, n + count);
  p->offA.assign(count + 1, 0);
  p->offS.assign(count + 1, 0);
  p->offU.assign(count + 1, 0);
  p->offV.assign(count + 1, 0);
  std::vector<BatchItem> items(count);
  std::vector<double> cost(count);
  int64_t wa = 0, wv = 0;
  bj_layout(count, m, n, items.data(), cost.data(), p->offA.data(), p->offS.data(),
            p->offU.data(), p->offV.data(), wa, wv);
  for (int k = 0; k < count; ++k) p->work += cost[k];
  p->work_elems_a = (size_t)round_up(wa, 64);
  p->work_elems_v = (size_t)round_up(wv, 64);
  p->order.resize(count);
  std::iota(p->order.begin(), p->order.end(), 0);
  std::stable_sort(p->order.begin(), p->order.end(),
                   [&](int x, int y) { return cost[x] > cost[y]; });

  DDC_HIP(hipGetDevice(&p->dev));
  DDC_HIP(hipDeviceGetAttribute(&p->cus, hipDeviceAttributeMultiprocessorCount, p->dev));
  if (p->cus < 1) p->cus = 1;
  const size_t order_len = p->order.size();
  if (hipMalloc(&p->d_items, sizeof(BatchItem) * count) != hipSuccess ||
      hipMalloc(&p->d_order, sizeof(int) * order_len) != hipSuccess ||
      hipMalloc(&p->d_counter, sizeof(int) * 64) != hipSuccess ||
      hipMalloc(&p->d_work, es * (p->work_elems_a + p->work_elems_v)) != hipSuccess) {
    (void)hipGetLastError();
    report_error("device allocation for the batch failed");
    return DDC_E_NOMEM;
  }
  std::vector<int> ord(p->order);
  DDC_HIP(hipMemcpy(p->d_items, items.data(), sizeof(BatchItem) * count, hipMemcpyHostToDevice));
  DDC_HIP(hipMemcpy(p->d_order, ord.data(), sizeof(int) * order_len, hipMemcpyHostToDevice));
  DDC_HIP(hipMemset(p->d_counter, 0, sizeof(int) * 64));
  DDC_HIP(hipStreamCreateWithFlags(&p->cap, hipStreamNonBlocking));
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto f = g_tune_cache.find(tune_key(p));
    if (f != g_tune_cache.end()) {
      p->cfg.variant = bj_variant(p);
      p->cfg.wgs = 1;
      p->cfg.coop_nt = f->second;
    }
  }
  return DDC_OK;
}

static int bj_run(svd_gpu_batch* p, const void* dA, void* dS, void* dU, void* dV, int* info,
                  hipStream_t st) {
  if (p->cfg.variant < 0) DDC_TRY(bj_tune(p, dA, dS, dU, dV, st));
  const bool same = p->exec && p->gA == dA && p->gS == dS && p->gU == dU && p->gV == dV &&
                    p->ginfo == info;
  if (!same) {
    if (p->exec) (void)hipGraphExecDestroy(p->exec);
    if (p->graph) (void)hipGraphDestroy(p->graph);
    p->exec = nullptr;
    p->graph = nullptr;
    DDC_HIP(hipStreamBeginCapture(p->cap, hipStreamCaptureModeThreadLocal));
    const int rc = bj_enqueue(p, p->cfg, dA, dS, dU, dV, info, p->cap);
    hipGraph_t gr = nullptr;
    const hipError_t e = hipStreamEndCapture(p->cap, &gr);
    if (rc) {
      if (gr) (void)hipGraphDestroy(gr);
      return rc;
    }
    DDC_HIP(e);
    p->graph = gr;
    DDC_HIP(hipGraphInstantiate(&p->exec, p->graph, nullptr, nullptr, 0));
    p->gA = dA;
    p->gS = dS;
    p->gU = dU;
    p->gV = dV;
    p->ginfo = info;
  }
  DDC_HIP(hipGraphLaunch(p->exec, st));
  return DDC_OK;
}

// ---------------------------------------------------------------------------
// The variant that allocates nothing: every buffer beyond the caller's inputs
// and outputs (matrix descriptors, processing order, queue head, working
// copies) lives in one file-scope device array, and the host-side
// descriptors in file-scope host arrays.  Each GPU holds its own copy of the
// device array (its address is looked up once per device); calls on one GPU
// share it, so calls that overlap on one GPU race.
// ---------------------------------------------------------------------------
constexpr size_t BJ_NA_BYTES = (size_t)32 << 20;  // device scratch per GPU
constexpr int BJ_NA_MAXCOUNT = 4096;              // matrices per call
constexpr int BJ_NA_MAXDEV = 64;
// fixed launch configuration: variant 1 (column blocks of 4), one workgroup
// per CU, whole-workgroup factorization from min(m, n) = 32 on
static const BjConfig kNoallocConfig = {1, 1, 32};

static __device__ __align__(256) char scratch[BJ_NA_BYTES];

namespace {
std::mutex g_na_mu;
char* g_na_ptr[BJ_NA_MAXDEV] = {};
int g_na_cus[BJ_NA_MAXDEV] = {};
BatchItem g_na_items[BJ_NA_MAXCOUNT];
double g_na_cost[BJ_NA_MAXCOUNT];
int g_na_order[BJ_NA_MAXCOUNT];
}  // namespace

static size_t na_align(size_t b) { return (b + 255) & ~(size_t)255; }

static int bj_noalloc(int count, const int* m, const int* n, int dtype, const void* dA, void* dS,
                      void* dU, void* dV, int* info, hipStream_t st) {
  int dev = 0;
  DDC_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= BJ_NA_MAXDEV) {
    report_error("device index beyond the no-alloc table");
    return DDC_E_ARG;
  }
  if (!g_na_ptr[dev]) {
    // set-up, once per device with that device current: the device address
    // of this GPU's copy of the scratch array (the array's name in host
    // code is only a host-side handle)
    void* ptr = nullptr;
    DDC_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    int cus = 0;
    DDC_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    g_na_cus[dev] = cus > 0 ? cus : 1;
    g_na_ptr[dev] = (char*)ptr;
  }
  char* base = g_na_ptr[dev];
  const size_t es = dtype == SVD_GPU_F64 ? 8 : 4;
  int64_t wa = 0, wv = 0;
  bj_layout(count, m, n, g_na_items, g_na_cost, nullptr, nullptr, nullptr, nullptr, wa, wv);
  const size_t b_items = na_align(sizeof(BatchItem) * count);
  const size_t b_order = na_align(sizeof(int) * count);
  const size_t b_ctr = 256;
  const size_t ea = (size_t)round_up(wa, 64), ev = (size_t)round_up(wv, 64);
  const size_t need = b_items + b_order + b_ctr + na_align(es * (ea + ev));
  if (need > BJ_NA_BYTES) {
    char msg[160];
    snprintf(msg, sizeof(msg), "batch needs %zu bytes of scratch; the no-alloc limit is %zu",
             need, BJ_NA_BYTES);
    report_error(msg);
    return DDC_E_ARG;
  }
  for (int k = 0; k < count; ++k) g_na_order[k] = k;
  // largest first, ties by index (std::sort works in place)
  std::sort(g_na_order, g_na_order + count, [](int x, int y) {
    return g_na_cost[x] > g_na_cost[y] || (g_na_cost[x] == g_na_cost[y] && x < y);
  });
  BatchItem* d_items = (BatchItem*)base;
  int* d_order = (int*)(base + b_items);
  int* d_ctr = (int*)(base + b_items + b_order);
  char* d_work = base + b_items + b_order + b_ctr;
  DDC_HIP(hipMemcpyAsync(d_items, g_na_items, sizeof(BatchItem) * count, hipMemcpyHostToDevice,
                         st));
  DDC_HIP(hipMemcpyAsync(d_order, g_na_order, sizeof(int) * count, hipMemcpyHostToDevice, st));
  // the host arrays are reused by the next call
  DDC_HIP(hipStreamSynchronize(st));
  // the queue head starts at zero (a fill kernel; the array keeps the last
  // call's contents)
  hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(64), 0, st, d_ctr, 0, 1);
  DDC_LAUNCHED();
  if (dtype == SVD_GPU_F64) {
    BjArgs<double> a;
    a.count = count;
    a.items = d_items;
    a.order = d_order;
    a.counter = d_ctr;
    a.A = (const double*)dA;
    a.S = (double*)dS;
    a.U = (double*)dU;
    a.V = (double*)dV;
    a.W = (double*)d_work;
    a.WV = (double*)d_work + ea;
    a.info = info;
    return bj_launch<double>(kNoallocConfig, g_na_cus[dev], a, st);
  }
  BjArgs<float> a;
  a.count = count;
  a.items = d_items;
  a.order = d_order;
  a.counter = d_ctr;
  a.A = (const float*)dA;
  a.S = (float*)dS;
  a.U = (float*)dU;
  a.V = (float*)dV;
  a.W = (float*)d_work;
  a.WV = (float*)d_work + ea;
  a.info = info;
  return bj_launch<float>(kNoallocConfig, g_na_cus[dev], a, st);
}

}  // namespace ddc

using namespace ddc;

extern "C" {

int svd_gpu_batched_plan(svd_gpu_batch** plan, int count, const int* m, const int* n, int dtype) {
  clear_error();
  if (!plan) {
    report_error("null plan pointer");
    return DDC_E_ARG;
  }
  *plan = nullptr;
  if (count < 1 || !m || !n || (dtype != SVD_GPU_F64 && dtype != SVD_GPU_F32)) {
    report_error("invalid batch arguments");
    return DDC_E_ARG;
  }
  for (int k = 0; k < count; ++k)
    if (m[k] < 1 || n[k] < 1 || m[k] > BJ_MAXDIM || n[k] > BJ_MAXDIM) {
      report_error("batched matrices need 1 <= m, n <= 256");
      return DDC_E_ARG;
    }
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) {
    report_error("no HIP device available");
    return DDC_E_NODEV;
  }
  svd_gpu_batch* p = new (std::nothrow) svd_gpu_batch;
  if (!p) return DDC_E_NOMEM;
  const int rc = bj_plan(p, count, m, n, dtype);
  if (rc) {
    bj_free(p);
    delete p;
    return rc;
  }
  *plan = p;
  return DDC_OK;
}

int svd_gpu_batched_offsets(const svd_gpu_batch* plan, long long* offA, long long* offS,
                            long long* offU, long long* offV) {
  if (!plan) return DDC_E_ARG;
  const size_t c = (size_t)plan->count + 1;
  if (offA) std::memcpy(offA, plan->offA.data(), c * sizeof(long long));
  if (offS) std::memcpy(offS, plan->offS.data(), c * sizeof(long long));
  if (offU) std::memcpy(offU, plan->offU.data(), c * sizeof(long long));
  if (offV) std::memcpy(offV, plan->offV.data(), c * sizeof(long long));
  return DDC_OK;
}

int svd_gpu_batched_tune(svd_gpu_batch* plan, const void* dA, void* dsigma, void* dU, void* dV,
                         void* stream) {
  clear_error();
  if (!plan || !dA || !dsigma || !dU || !dV) {
    report_error("invalid batch arguments");
    return DDC_E_ARG;
  }
  std::lock_guard<std::mutex> lk(plan->mu);
  return bj_tune(plan, dA, dsigma, dU, dV, (hipStream_t)stream);
}

int svd_gpu_batched_set_config(svd_gpu_batch* plan, int variant, int wgs_per_cu,
                               int coop_min_n) {
  clear_error();
  if (!plan || variant < 0 || variant >= kNumVariants || wgs_per_cu < 1 || wgs_per_cu > 8 ||
      coop_min_n < 1) {
    report_error("invalid batch configuration");
    return DDC_E_ARG;
  }
  std::lock_guard<std::mutex> lk(plan->mu);
  plan->cfg.variant = variant;
  plan->cfg.wgs = wgs_per_cu;
  plan->cfg.coop_nt = coop_min_n;
  plan->gA = nullptr;  // forces a new graph
  plan->ginfo = nullptr;
  if (plan->exec) (void)hipGraphExecDestroy(plan->exec);
  plan->exec = nullptr;
  return DDC_OK;
}

int svd_gpu_batched_config(const svd_gpu_batch* plan, int* variant, int* wgs_per_cu,
                           int* coop_min_n, int* block_small, int* block_large) {
  if (!plan) return DDC_E_ARG;
  const BjConfig& c = plan->cfg;
  if (variant) *variant = c.variant;
  if (wgs_per_cu) *wgs_per_cu = c.wgs;
  if (coop_min_n) *coop_min_n = c.coop_nt;
  if (block_small) *block_small = c.variant >= 0 ? kVariants[c.variant].b12 : 0;
  if (block_large) *block_large = c.variant >= 0 ? kVariants[c.variant].b34 : 0;
  return kNumVariants;
}

int svd_gpu_batched_run(svd_gpu_batch* plan, const void* dA, void* dsigma, void* dU, void* dV,
                        int* dinfo, void* stream) {
  clear_error();
  if (!plan || !dA || !dsigma || !dU || !dV) {
    report_error("invalid batch arguments");
    return DDC_E_ARG;
  }
  std::lock_guard<std::mutex> lk(plan->mu);
  return bj_run(plan, dA, dsigma, dU, dV, dinfo, (hipStream_t)stream);
}

int svd_gpu_batched_noalloc(int count, const int* m, const int* n, int dtype, const void* dA,
                            void* dsigma, void* dU, void* dV, int* dinfo, void* stream) {
  clear_error();
  if (count < 1 || count > BJ_NA_MAXCOUNT || !m || !n || !dA || !dsigma || !dU || !dV ||
      (dtype != SVD_GPU_F64 && dtype != SVD_GPU_F32)) {
    report_error("invalid batch arguments (1 <= count <= 4096 for the no-alloc entry point)");
    return DDC_E_ARG;
  }
  for (int k = 0; k < count; ++k)
    if (m[k] < 1 || n[k] < 1 || m[k] > BJ_MAXDIM || n[k] > BJ_MAXDIM) {
      report_error("batched matrices need 1 <= m, n <= 256");
      return DDC_E_ARG;
    }
  std::lock_guard<std::mutex> lk(g_na_mu);
  return bj_noalloc(count, m, n, dtype, dA, dsigma, dU, dV, dinfo, (hipStream_t)stream);
}

void svd_gpu_batched_destroy(svd_gpu_batch* plan) {
  if (!plan) return;
  {
    std::lock_guard<std::mutex> lk(plan->mu);
    bj_free(plan);
  }
  delete plan;
}

}  // extern "C"
