// householder.h -- device pieces shared by the bidiagonalization kernels:
// the Householder data of a vector and wave sums on DPP and lane swaps.
#pragma once

#include "ddc_common.h"

namespace ddc {

// Householder data of the vector x with |x|^2 = sumsq and first entry x1,
// as the reference forms it (update_scale_matcol.cl:58-82): diag =
// -sign(x1)|x|, reflector = (x + sign(x1)|x| e1) / rl with
// rl = sqrt(2) sqrt(|x|^2 + ||x| x1|).  A zero vector gives rl = 0 and is
// treated as "no reflection" (the reference divides by zero there).
struct Refl {
  double nrm, sgn, rl;
  __device__ __forceinline__ void make(double sumsq, double x1) {
    nrm = sqrt(sumsq);
    sgn = (x1 < 0) ? -1.0 : 1.0;
    rl = sqrt(2.0) * sqrt(nrm * nrm + fabs(nrm * x1));
  }
  __device__ __forceinline__ double diag() const { return rl != 0.0 ? -sgn * nrm : 0.0; }
  __device__ __forceinline__ double vec(double x, bool first) const {
    if (rl == 0.0) return 0.0;
    return (first ? x + sgn * nrm : x) / rl;
  }
  // (w^T reflector) from (w^T x) and the first entry w1 of w
  __device__ __forceinline__ double dot(double wx, double w1) const {
    return rl != 0.0 ? (wx + sgn * nrm * w1) / rl : 0.0;
  }
};

// num / d from ir = 1/d (0 for d = 0, giving 0): q0 = num ir, then one
// correction q0 + (num - q0 d) ir with fused multiply-adds.
__device__ __forceinline__ double rl_quot(double num, double d, double ir) {
  const double q0 = num * ir;
  return fma(fma(-q0, d, num), ir, q0);
}

// Wave sum by DPP (row-local butterflies, then the row broadcasts of gfx9),
// in a fixed order; every lane gets lane 63's total.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_take(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, ROWS, 0xf, false);
  return __builtin_bit_cast(double, ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}
// (every lane written: no old value to set)
template <int CTRL>
__device__ __forceinline__ double dpp_all(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)b, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, false);
  return __builtin_bit_cast(double, ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}
constexpr int DPP_XOR1 = 0xB1;          // quad_perm [1,0,3,2]
constexpr int DPP_XOR2 = 0x4E;          // quad_perm [2,3,0,1]
constexpr int DPP_QUAD_REVERSE = 0x1B;  // quad_perm [3,2,1,0]
constexpr int DPP_HALF_MIRROR = 0x141;  // lane i of eight from lane 7 - i
constexpr int DPP_MIRROR = 0x140;       // lane i of sixteen from lane 15 - i
constexpr int DPP_ROR8 = 0x128;         // rows of sixteen rotated by eight
constexpr int DPP_ROR4 = 0x124;         // and by four

// The value of lane l, wave-uniform.
__device__ __forceinline__ double lane_value(double v, int l) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)b, l);
  const unsigned hi = __builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ double lane63(double v) { return lane_value(v, 63); }
__device__ __forceinline__ double wave_total(double v) {
  v += dpp_all<DPP_XOR1>(v);         // pairs
  v += dpp_all<DPP_XOR2>(v);         // quads
  v += dpp_all<DPP_HALF_MIRROR>(v);  // eights
  v += dpp_all<DPP_MIRROR>(v);       // rows of 16
  v += dpp_take<0x142, 0xA>(v);      // row_bcast:15 into rows 1, 3
  v += dpp_take<0x143, 0xC>(v);      // row_bcast:31 into rows 2, 3: lane 63 has the total
  return lane63(v);
}
// Three wave totals with their stages interleaved (independent chains).
__device__ __forceinline__ void wave_total3(double& a, double& b, double& c) {
  a += dpp_all<DPP_XOR1>(a);
  b += dpp_all<DPP_XOR1>(b);
  c += dpp_all<DPP_XOR1>(c);
  a += dpp_all<DPP_XOR2>(a);
  b += dpp_all<DPP_XOR2>(b);
  c += dpp_all<DPP_XOR2>(c);
  a += dpp_all<DPP_HALF_MIRROR>(a);
  b += dpp_all<DPP_HALF_MIRROR>(b);
  c += dpp_all<DPP_HALF_MIRROR>(c);
  a += dpp_all<DPP_MIRROR>(a);
  b += dpp_all<DPP_MIRROR>(b);
  c += dpp_all<DPP_MIRROR>(c);
  a += dpp_take<0x142, 0xA>(a);
  b += dpp_take<0x142, 0xA>(b);
  c += dpp_take<0x142, 0xA>(c);
  a += dpp_take<0x143, 0xC>(a);
  b += dpp_take<0x143, 0xC>(b);
  c += dpp_take<0x143, 0xC>(c);
  a = lane63(a);
  b = lane63(b);
  c = lane63(c);
}

// Exchange of lane halves between two registers: after swap_lanes<32>(a, b)
// a holds (a's lanes 0-31, b's lanes 0-31) and b (a's lanes 32-63, b's lanes
// 32-63); swap_lanes<16> does the same within each 32 lanes (gfx950
// v_permlane32_swap_b32 / v_permlane16_swap_b32).  With a = b = v the sum of
// the two results is the butterfly sum across the halves.
template <int W>
__device__ __forceinline__ void swap_lanes(double& a, double& b) {
  static_assert(W == 32 || W == 16, "halves of 64 or of 32 lanes");
  const unsigned long long x = __builtin_bit_cast(unsigned long long, a);
  const unsigned long long y = __builtin_bit_cast(unsigned long long, b);
  const unsigned xl = (unsigned)x, xh = (unsigned)(x >> 32);
  const unsigned yl = (unsigned)y, yh = (unsigned)(y >> 32);
  if constexpr (W == 32) {
    const auto l = __builtin_amdgcn_permlane32_swap(xl, yl, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(xh, yh, false, false);
    a = __builtin_bit_cast(double, ((unsigned long long)h[0] << 32) | l[0]);
    b = __builtin_bit_cast(double, ((unsigned long long)h[1] << 32) | l[1]);
  } else {
    const auto l = __builtin_amdgcn_permlane16_swap(xl, yl, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(xh, yh, false, false);
    a = __builtin_bit_cast(double, ((unsigned long long)h[0] << 32) | l[0]);
    b = __builtin_bit_cast(double, ((unsigned long long)h[1] << 32) | l[1]);
  }
}
template <int W>
__device__ __forceinline__ double half_sum(double v) {
  double a = v, b = v;
  swap_lanes<W>(a, b);
  return a + b;
}

// Wave sums of N values (N = 1, 2, 4, 8 or 16), value i delivered to the
// 64 / N lanes with lane / (64 / N) == i.  Each of the first log2 N stages
// halves the values a lane carries: two lane-swap stages, then DPP.
template <int N>
__device__ __forceinline__ double wave_scatter(double (&g)[N]) {
  static_assert(N == 1 || N == 2 || N == 4 || N == 8 || N == 16, "a power of two up to 16");
  const int lane = threadIdx.x & 63;
  if constexpr (N >= 2) {
#pragma unroll
    for (int j = 0; j < N / 2; ++j) {
      swap_lanes<32>(g[j], g[j + N / 2]);
      g[j] += g[j + N / 2];
    }
  }
  if constexpr (N >= 4) {
#pragma unroll
    for (int j = 0; j < N / 4; ++j) {
      swap_lanes<16>(g[j], g[j + N / 4]);
      g[j] += g[j + N / 4];
    }
  }
  if constexpr (N >= 8) {
    const bool up = (lane >> 3) & 1;
#pragma unroll
    for (int j = 0; j < N / 8; ++j) {
      const double lo = g[j], hi = g[j + N / 8];
      g[j] = (up ? hi : lo) + dpp_all<DPP_ROR8>(up ? lo : hi);
    }
  }
  if constexpr (N >= 16) {
    const bool up = (lane >> 2) & 1;
#pragma unroll
    for (int j = 0; j < N / 16; ++j) {
      const double lo = g[j], hi = g[j + N / 16];
      g[j] = (up ? hi : lo) + dpp_all<DPP_HALF_MIRROR>(up ? lo : hi);
    }
  }
  double v = g[0];
  v += dpp_all<DPP_XOR1>(v);
  v += dpp_all<DPP_XOR2>(v);
  if constexpr (N <= 8) v += dpp_all<DPP_HALF_MIRROR>(v);
  if constexpr (N <= 4) v += dpp_all<DPP_MIRROR>(v);
  if constexpr (N <= 2) v = half_sum<16>(v);
  if constexpr (N <= 1) v = half_sum<32>(v);
  return v;
}

}  // namespace ddc
