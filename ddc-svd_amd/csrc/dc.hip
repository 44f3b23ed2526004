// dc.hip -- singular values of an upper bidiagonal by divide and conquer, FP64.
//
// Replaces GetSingularValues_Parallel (Calculations-Parallel.c:852-874) and
// its recursion (DivideAndConquer_Parallel :706-850).  The split is the
// reference's: B is N x (N+1) with diagonal a and super-diagonal b, row
// K = N/2 is removed, the children are K x (K+1) and (N-K-1) x (N-K), and
// each merge needs only the first and last rows of the children's right
// singular vector matrices (the Konda-Nakamura values-only form).
//
// What differs from the reference is the numerical core of a merge:
//  * relative deflation (|z_j| or pole gaps below 8 eps scale) with Givens
//    rotations of the first/last rows, instead of the absolute thresholds
//    1e-14/1e-20 (:143-144, :467);
//  * each secular root is bracketed between its poles and found by
//    interpolation, safeguarded by bisection, in the offset tau from the nearer
//    pole, so sigma - d_j is formed without cancellation and no step can jump
//    to a neighbouring root (the reference's duplicate-root failure, :163-254);
//  * the first/last rows come from the Gu-Eisenstat z-hat (:445-465 uses a
//    log-domain product with the same role), evaluated from the stored
//    offsets.
//
// GPU mapping: the recursion tree depends on n alone.  Its nodes are named by
// their place in a binary heap (children of id: 2 id, 2 id + 1), from which
// every work-group finds its own range by walking down from the root (at most
// log2 n integer steps): no table is built on the host or copied, which was
// three copies, a stream synchronization and 110 us before the first kernel.
// The tree is processed bottom-up, one depth per round; the ranges of a depth
// differ by at most one entry.  Per depth five kernels run over all its
// merges: prep (one work-group per merge: rank-merge of the two
// sorted child spectra, deflation, compaction), roots (one wave per root),
// zhat (one wave per pole), rows (one wave per root: first/last rows of the
// new singular vectors) and assemble (one work-group per merge); depths of
// ranges up to DC_SMALL do all five in one launch.  The roots
// kernel gives a whole wave to each root: its lanes split the O(K) secular
// sum, so the top merge of an n = 8192 problem fills the GPU.
#include <algorithm>

#include "ddc_common.h"
#include "householder.h"

namespace ddc {

constexpr double EPS = 2.220446049250313e-16;
// Ranges up to here take one launch per depth (dc_small).  The stage at
// n = 64, 256 and 1187, in us: 145, 218, 398 with none, 134, 200, 372 up to 8,
// 140, 205, 371 up to 16, 179, 248, 385 up to 32.
constexpr int DC_SMALL = 8;
constexpr double TINY = 2.2250738585072014e-308;

// A node of the tree: positions [off, off+N), split row off+K; a merge if
// N >= 2, else a leaf.
struct DcMerge {
  int off, N, K;
  int c1, c2;  // children's ids
};

// The node at heap place id (1 the root) of the tree over n entries; false
// if the tree has none there (an ancestor is a leaf).
__device__ __forceinline__ bool dc_node(int n, int id, DcMerge& M) {
  int off = 0, N = n;
  for (int b = 30 - __builtin_clz(id); b >= 0; --b) {
    if (N < 2) return false;
    const int K = N / 2;
    if ((id >> b) & 1) {
      off += K + 1;
      N -= K + 1;
    } else {
      N = K;
    }
  }
  M = DcMerge{off, N, N / 2, 2 * id, 2 * id + 1};
  return true;
}

// Per-merge scalars produced by prep.
struct DcMergeState {
  int kept;          // K': non-deflated poles, including the pole at 0
  double scale;      // poles and z are divided by it in the secular solve
  double znorm;      // |z| (scaled)
  double cg, sg;     // rotation of the two null columns
};

struct DcBufs {
  double *a, *b;                 // inputs
  double *sig, *fr, *lr;         // node outputs at node positions
  double *phi, *psi;             // per node, by id
  double *wd, *wz, *wF, *wL;     // sorted merged data
  int* flag;                     // 1 = deflated
  double *kd, *kz, *kF, *kL;     // kept (scaled poles/z)
  double *dd, *dF, *dL;          // deflated (unscaled poles)
  int* org;                      // root origin (index into kept)
  double* tau;                   // root offset from its origin pole (scaled)
  double* zh;                    // z-hat
  double *fn, *ln;               // new first/last rows for the roots
  DcMergeState* ms;              // per merge, by id
  int n;                         // entries of the whole tree
  double* out;                   // final singular values
};

// ---------------------------------------------------------------------------
// leaves: N == 1 ([a b], sigma = hypot) and N == 0 (W = [1])
// ---------------------------------------------------------------------------
__global__ void dc_leaves(DcBufs B, int ids) {
  const int node = 1 + blockIdx.x * blockDim.x + threadIdx.x;
  DcMerge M;
  if (node > ids || !dc_node(B.n, node, M) || M.N >= 2) return;
  const int off = M.off, N = M.N;
  if (N == 0) {
    B.phi[node] = 1.0;
    B.psi[node] = 1.0;
    return;
  }
  double a = B.a[off], b = B.b[off];
  double s = hypot(a, b);
  B.sig[off] = s;
  if (s == 0.0) {
    B.fr[off] = 1.0;
    B.lr[off] = 0.0;
    B.phi[node] = 0.0;
    B.psi[node] = 1.0;
  } else {
    // right singular vector (a, b)/s, null vector (-b, a)/s
    B.fr[off] = a / s;
    B.lr[off] = b / s;
    B.phi[node] = -b / s;
    B.psi[node] = a / s;
  }
}

// ---------------------------------------------------------------------------
// helpers for one work-group of 256 threads
// ---------------------------------------------------------------------------
__device__ __forceinline__ int count_less(const double* x, int n, double v) {
  int lo = 0, hi = n;
  while (lo < hi) {
    int mid = (lo + hi) >> 1;
    if (x[mid] < v) lo = mid + 1; else hi = mid;
  }
  return lo;
}
__device__ __forceinline__ int count_leq(const double* x, int n, double v) {
  int lo = 0, hi = n;
  while (lo < hi) {
    int mid = (lo + hi) >> 1;
    if (x[mid] <= v) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// Exclusive scan of per-thread counts over the 256-thread group.
__device__ int group_exscan(int v, int* tmp, int* total) {
  int tid = threadIdx.x;
  tmp[tid] = v;
  __syncthreads();
  for (int o = 1; o < 256; o <<= 1) {
    int add = (tid >= o) ? tmp[tid - o] : 0;
    __syncthreads();
    tmp[tid] += add;
    __syncthreads();
  }
  int incl = tmp[tid];
  *total = tmp[255];
  __syncthreads();
  return incl - v;
}

__device__ double group_max(double v, double* red) {
  v = fmax(v, __shfl_xor(v, 32, 64));
  v = fmax(v, __shfl_xor(v, 16, 64));
  v = fmax(v, __shfl_xor(v, 8, 64));
  v = fmax(v, __shfl_xor(v, 4, 64));
  v = fmax(v, __shfl_xor(v, 2, 64));
  v = fmax(v, __shfl_xor(v, 1, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double r = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
  __syncthreads();
  return r;
}

// ---------------------------------------------------------------------------
// prep: build the merged arrow, sort, deflate, compact.  One group per merge.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void prep_merge(const DcBufs& B, int id, const DcMerge& M) {
  __shared__ double red[4];
  __shared__ int tmp[256];
  __shared__ double s_tol, s_scale;
  __shared__ int s_total;
  const int tid = threadIdx.x;
  const int off = M.off, N = M.N, K = M.K, N2 = N - K - 1;
  const double* s1 = B.sig + off;
  const double* f1 = B.fr + off;
  const double* l1 = B.lr + off;
  const double* s2 = B.sig + off + K + 1;
  const double* f2 = B.fr + off + K + 1;
  const double* l2 = B.lr + off + K + 1;
  const double aK = B.a[off + K], bK = B.b[off + K];
  const double ph1 = B.phi[M.c1], ps1 = B.psi[M.c1];
  const double ph2 = B.phi[M.c2], ps2 = B.psi[M.c2];
  const double x = aK * ps1, y = bK * ph2;
  const double r0 = hypot(x, y);
  const double cg = (r0 > 0.0) ? x / r0 : 1.0;
  const double sg = (r0 > 0.0) ? y / r0 : 0.0;

  double* wd = B.wd + off;
  double* wz = B.wz + off;
  double* wF = B.wF + off;
  double* wL = B.wL + off;
  int* flag = B.flag + off;

  // 1. merge the two ascending child spectra behind the pole at 0 (on ties
  // the first child's value first).  Merge path: thread t writes the merged
  // outputs [t per, (t+1) per), finding its start in the two lists by one
  // binary search and then walking both (a binary search per element was a
  // chain of 13 dependent loads per element, most of this kernel's time).
  double zmax = 0.0;
  if (tid == 0) {
    wd[0] = 0.0;
    wz[0] = r0;
    wF[0] = cg * ph1;
    wL[0] = sg * ps2;
    zmax = fabs(r0);
  }
  {
    const int NO = K + N2;  // merged outputs after the pole
    const int per = (NO + 255) / 256;
    const int d0 = min(NO, tid * per), d1 = min(NO, d0 + per);
    int lo = max(0, d0 - N2), hi = min(d0, K);
    while (lo < hi) {  // i = the number of first-child values among outputs < d0
      const int mid = (lo + hi) >> 1;
      if (s1[mid] <= s2[d0 - mid - 1]) lo = mid + 1;
      else hi = mid;
    }
    int i = lo, j = d0 - lo;
    for (int p = d0; p < d1; ++p) {
      const bool first = j >= N2 || (i < K && s1[i] <= s2[j]);
      if (first) {
        const double zv = aK * l1[i];
        wd[1 + p] = s1[i];
        wz[1 + p] = zv;
        wF[1 + p] = f1[i];
        wL[1 + p] = 0.0;
        zmax = fmax(zmax, fabs(zv));
        ++i;
      } else {
        const double zv = bK * f2[j];
        wd[1 + p] = s2[j];
        wz[1 + p] = zv;
        wF[1 + p] = 0.0;
        wL[1 + p] = l2[j];
        zmax = fmax(zmax, fabs(zv));
        ++j;
      }
    }
  }
  zmax = group_max(zmax, red);
  __syncthreads();
  if (tid == 0) {
    double dmax = (N > 1) ? wd[N - 1] : 0.0;
    double sc = fmax(dmax, zmax);
    s_scale = sc;
    s_tol = fmax(8.0 * EPS * sc, TINY);
  }
  __syncthreads();
  const double tol = s_tol;

  // 2. deflate negligible z_j (j >= 1)
  for (int j = tid; j < N; j += 256) flag[j] = (j >= 1 && fabs(wz[j]) <= tol) ? 1 : 0;
  __syncthreads();

  // 3. close poles: sequential rotations along the sorted kept entries.
  // Chains of close poles are rare; one thread walks the list, and only if
  // some kept entry lies within tol of its predecessor in the sorted list
  // (else no pair of kept entries is that close and the walk rotates
  // nothing).
  int close = 0;
  for (int j = 1 + tid; j < N; j += 256) close |= (!flag[j] && wd[j] - wd[j - 1] <= tol) ? 1 : 0;
  close = __syncthreads_or(close);
  if (tid == 0 && close) {
    int prev = 0;
    for (int j = 1; j < N; ++j) {
      if (flag[j]) continue;
      double dj = wd[j];
      if (dj - wd[prev] <= tol) {
        double zp = wz[prev], zj = wz[j];
        double r = hypot(zp, zj);
        if (prev == 0) {
          // pole ~0: fold z_j into z_0, deflate j (its value is ~0)
          double c = zp / r, s = zj / r;
          double F0 = wF[0], Fj = wF[j], L0 = wL[0], Lj = wL[j];
          wF[0] = c * F0 + s * Fj;
          wF[j] = -s * F0 + c * Fj;
          wL[0] = c * L0 + s * Lj;
          wL[j] = -s * L0 + c * Lj;
          wz[0] = r;
          wz[j] = 0.0;
          flag[j] = 1;
          continue;
        }
        double c = zj / r, s = zp / r;
        double Fp = wF[prev], Fj = wF[j], Lp = wL[prev], Lj = wL[j];
        wF[prev] = c * Fp - s * Fj;
        wF[j] = s * Fp + c * Fj;
        wL[prev] = c * Lp - s * Lj;
        wL[j] = s * Lp + c * Lj;
        wz[prev] = 0.0;
        wz[j] = r;
        flag[prev] = 1;
      }
      prev = j;
    }
  }
  // a zero arrow (every pole and z at zero) keeps its root at zero
  if (tid == 0 && fabs(wz[0]) <= tol) wz[0] = s_scale > 0.0 ? tol : 0.0;
  __syncthreads();

  // 4. compaction: kept entries to [0, K'), deflated to [0, N-K') in order
  const int per = (N + 255) / 256;
  const int b0 = min(N, tid * per), b1 = min(N, b0 + per);
  int nk = 0;
  for (int j = b0; j < b1; ++j) nk += flag[j] ? 0 : 1;
  int kept_tot = 0;
  int kpos = group_exscan(nk, tmp, &kept_tot);
  if (tid == 0) s_total = kept_tot;
  __syncthreads();
  const int kept = s_total;
  const double sc = s_scale;
  const double isc = (sc > 0.0) ? 1.0 / sc : 1.0;
  int dpos = b0 - kpos;
  for (int j = b0; j < b1; ++j) {
    if (!flag[j]) {
      B.kd[off + kpos] = wd[j] * isc;
      B.kz[off + kpos] = wz[j] * isc;
      B.kF[off + kpos] = wF[j];
      B.kL[off + kpos] = wL[j];
      ++kpos;
    } else {
      B.dd[off + dpos] = wd[j];
      B.dF[off + dpos] = wF[j];
      B.dL[off + dpos] = wL[j];
      ++dpos;
    }
  }
  // |z| of the kept (scaled) entries
  double zz = 0.0;
  __syncthreads();
  for (int q = tid; q < kept; q += 256) {
    double v = B.kz[off + q];
    zz += v * v;
  }
  zz = wave_total(zz);
  if ((tid & 63) == 0) red[tid >> 6] = zz;
  __syncthreads();
  if (tid == 0) {
    DcMergeState st;
    st.kept = kept;
    st.scale = (sc > 0.0) ? sc : 1.0;
    st.znorm = sqrt(red[0] + red[1] + red[2] + red[3]);
    st.cg = cg;
    st.sg = sg;
    B.ms[id] = st;
    B.phi[id] = -sg * ph1;
    B.psi[id] = cg * ps2;
  }
}

// Wave-cooperative secular function f = 1 + psi + phi at w = d_o + tau, with
// g_j = (d_j - w)(d_j + w), psi the sum of z_j^2 / g_j over j <= split and phi
// over the rest, and their derivatives by w^2 (sums of z_j^2 / g_j^2): lane l
// takes j = l, l+64, ...; a fixed-order wave sum, the same in every lane.
struct Secular {
  double psi, phi, dpsi, dphi;
};
__device__ __forceinline__ Secular secular_wave(const double* d, const double* z, int K, int split,
                                                int o, double tau, int lane) {
  const double dO = d[o];
  double ps = 0.0, ph = 0.0, dps = 0.0, dph = 0.0;
  for (int j = lane; j < K; j += 64) {
    const double zj = z[j];
    const double dj = d[j];
    const double ig = 1.0 / (((dj - dO) - tau) * (dj + dO + tau));
    const double t = (zj * zj) * ig, dt = t * ig;
    const bool low = j <= split;
    ps += low ? t : 0.0;
    dps += low ? dt : 0.0;
    ph += low ? 0.0 : t;
    dph += low ? 0.0 : dt;
  }
  Secular r;
  r.psi = wave_total(ps);
  r.phi = wave_total(ph);
  r.dpsi = wave_total(dps);
  r.dphi = wave_total(dph);
  return r;
}

__device__ __forceinline__ double wave_prod(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v *= __shfl_xor(v, o, 64);
  return v;
}

// ---------------------------------------------------------------------------
// roots: one wave per secular root
// ---------------------------------------------------------------------------
__device__ __forceinline__ void root_item(const DcBufs& B, int id, const DcMerge& M, int item,
                                         int lane) {
  const DcMergeState st = B.ms[id];
  const int i = item;
  const int K = st.kept;
  if (i >= K) return;
  const double* d = B.kd + M.off;
  const double* z = B.kz + M.off;
  if (K == 1) {
    if (lane == 0) {
      B.org[M.off] = 0;
      B.tau[M.off] = fabs(z[0]);
    }
    return;
  }
  // The root lies between the poles pa and pb (the last one beyond pb); it
  // is found as an offset from the nearer pole o, u = |tau| in (lo, hi].  The
  // sign of f at the middle tells which pole that is.
  const bool last = i == K - 1;
  const int pa = last ? i - 1 : i, pb = pa + 1;
  int o = i;
  double hi = st.znorm, sgn = 1.0;
  Secular f;
  double t;
  if (!last) {
    const double mid = 0.5 * (d[i] + d[i + 1]);
    f = secular_wave(d, z, K, pa, i, mid - d[i], lane);
    if (1.0 + f.psi + f.phi < 0.0) {
      o = i + 1;
      sgn = -1.0;
    }
    hi = fabs(mid - d[o]);
    t = hi;
  } else {
    t = 0.5 * hi;
    f = secular_wave(d, z, K, pa, o, t, lane);
  }
  // Each step replaces psi and phi by one pole each, at d_pa^2 and d_pb^2,
  // that match their values and slopes (R.-C. Li's "middle way", Solving
  // Secular Equations Stably and Efficiently, LAPACK Working Note 89, 1993),
  // and takes the root of the quadratic that is left; a
  // step against the sign of f is replaced by Newton's.  Every evaluation
  // narrows the bracket by the sign of f, and an iterate outside it by
  // bisection (geometric while it spans a factor above four, as the roots lie
  // at any relative offset from the pole).  Stops when the step or the
  // bracket is at the rounding level of u or f at that of its own sum: no
  // later sign would be more than rounding, and following them to the last
  // bit by bisection was most of the time.  Over 60 bidiagonals (random,
  // Gaussian, constant, graded) the values' errors are those of that search
  // within 5%.  With the tree found on the device the stage went from 0.35 to
  // 0.15 ms at n = 64 and from 1.0 to 0.40 ms at n = 1187 (0.13 and 0.37 with
  // dc_small).
  const double dO = d[o], dA = d[pa], dB = d[pb];
  double lo = 0.0, res = -1.0;
  for (int itn = 0; itn < 400; ++itn) {
    const double fx = 1.0 + f.psi + f.phi, fa = 1.0 + (f.phi - f.psi);
    if (fx == 0.0) {
      res = t;
      break;
    }
    // origin below the root: f < 0 -> root further out; origin above: f > 0.
    // The middle (t = hi) only bounds the bracket.
    if (t < hi) {
      if ((sgn > 0.0) ? (fx < 0.0) : (fx > 0.0)) lo = t;
      else hi = t;
      if (hi - lo <= 2.0 * EPS * lo) break;
    }
    const double w = dO + sgn * t, tau = sgn * t;
    const double ga = ((dA - dO) - tau) * (dA + w), gb = ((dB - dO) - tau) * (dB + w);
    const double c = fx - ga * f.dpsi - gb * f.dphi;
    const double a = (ga + gb) * fx - ga * gb * (f.dpsi + f.dphi);
    const double b = ga * gb * fx;
    const double s = sqrt(fmax(0.0, a * a - 4.0 * b * c));
    double eta;  // step in w^2
    if (last) eta = a < 0.0 ? 2.0 * b / (a - s) : (a + s) / (2.0 * c);
    else eta = a <= 0.0 ? (a - s) / (2.0 * c) : 2.0 * b / (a + s);
    if (!(fx * eta < 0.0)) eta = -fx / (f.dpsi + f.dphi);
    const double w2 = w * w + eta;
    const double du = w2 > 0.0 ? sgn * eta / (w + sqrt(w2)) : INFINITY;
    const double u = t + du;
    const bool in = u > lo && u < hi;
    if (fabs(fx) <= EPS * fa && fa < INFINITY) {
      res = in ? u : t;
      break;
    }
    if (fabs(du) <= 2.0 * EPS * t && in) {
      res = u;
      break;
    }
    if (in) t = u;
    else if (lo == 0.0) t = hi * 0.0625;
    else if (hi > 4.0 * lo) t = sqrt(lo * hi);
    else t = 0.5 * (lo + hi);
    if (!(t > lo && t < hi)) break;
    f = secular_wave(d, z, K, pa, o, sgn * t, lane);
  }
  if (lane == 0) {
    B.org[M.off + i] = o;
    B.tau[M.off + i] = sgn * (res > 0.0 ? res : 0.5 * (lo + hi));
  }
}

// ---------------------------------------------------------------------------
// zhat: one wave per kept pole.  zhat_j^2 = (w_{K-1}^2 - d_j^2)
//   * prod_{k<j} (w_k^2 - d_j^2)/(d_k^2 - d_j^2)
//   * prod_{j<=k<K-1} (w_k^2 - d_j^2)/(d_{k+1}^2 - d_j^2)
// with w_k - d_j = (d_{org(k)} - d_j) + tau_k.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void zhat_item(const DcBufs& B, int id, const DcMerge& M, int item,
                                         int lane) {
  const int K = B.ms[id].kept;
  const int j = item;
  if (j >= K) return;
  const double* d = B.kd + M.off;
  const int* org = B.org + M.off;
  const double* tau = B.tau + M.off;
  const double dj = d[j];
  double prod = 1.0;
  for (int k = lane; k < K - 1; k += 64) {
    double wm = (d[org[k]] - dj) + tau[k];  // w_k - d_j
    double wp = d[org[k]] + tau[k] + dj;    // w_k + d_j
    double dk = (k < j) ? d[k] : d[k + 1];
    prod *= (wm * wp) / ((dk - dj) * (dk + dj));
  }
  prod = wave_prod(prod);
  if (lane == 0) {
    double wm = (d[org[K - 1]] - dj) + tau[K - 1];
    double wp = d[org[K - 1]] + tau[K - 1] + dj;
    prod *= wm * wp;
    B.zh[M.off + j] = copysign(sqrt(fabs(prod)), B.kz[M.off + j]);
  }
}

// ---------------------------------------------------------------------------
// rows: one wave per root: first/last rows of the merged right vectors.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void row_item(const DcBufs& B, int id, const DcMerge& M, int item,
                                         int lane) {
  const int K = B.ms[id].kept;
  const int i = item;
  if (i >= K) return;
  const double* d = B.kd + M.off;
  const double* zh = B.zh + M.off;
  const double* F = B.kF + M.off;
  const double* L = B.kL + M.off;
  const int o = B.org[M.off + i];
  const double ti = B.tau[M.off + i];
  const double dO = d[o];
  const double w = dO + ti;
  double nn = 0.0, fs = 0.0, ls = 0.0;
  if (K > 1) {
    for (int j = lane; j < K; j += 64) {
      double v = zh[j] / (((d[j] - dO) - ti) * (d[j] + w));
      nn += v * v;
      fs += F[j] * v;
      ls += L[j] * v;
    }
    wave_total3(nn, fs, ls);
  }
  if (lane != 0) return;
  if (nn > 0.0 && isfinite(nn)) {
    double inv = 1.0 / sqrt(nn);
    B.fn[M.off + i] = fs * inv;
    B.ln[M.off + i] = ls * inv;
  } else {
    // a single kept pole (the arrow is 1 x 1) or a vector lost to
    // underflow: the singular vector is the pole's own unit vector
    B.fn[M.off + i] = F[o];
    B.ln[M.off + i] = L[o];
  }
}

// ---------------------------------------------------------------------------
// assemble: merge the ascending roots with the ascending deflated values.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void assemble_merge(const DcBufs& B, int id, const DcMerge& M) {
  const DcMergeState st = B.ms[id];
  const int off = M.off, N = M.N, K = st.kept, ND = N - K;
  const double* d = B.kd + off;
  const double* dd = B.dd + off;
  // roots: w_i = (d_o + tau_i) * scale
  for (int i = threadIdx.x; i < K; i += 256) {
    double w = (d[B.org[off + i]] + B.tau[off + i]) * st.scale;
    int pos = i + count_less(dd, ND, w);
    if (id == 1) {
      B.out[pos] = w;
    } else {
      B.sig[off + pos] = w;
      B.fr[off + pos] = B.fn[off + i];
      B.lr[off + pos] = B.ln[off + i];
    }
  }
  for (int q = threadIdx.x; q < ND; q += 256) {
    double v = dd[q];
    // ties go after the roots that equal v
    int lo = 0, hi = K;
    while (lo < hi) {
      int mid = (lo + hi) >> 1;
      double wm = (d[B.org[off + mid]] + B.tau[off + mid]) * st.scale;
      if (wm <= v) lo = mid + 1; else hi = mid;
    }
    int pos = q + lo;
    if (id == 1) {
      B.out[pos] = v;
    } else {
      B.sig[off + pos] = v;
      B.fr[off + pos] = B.dF[off + q];
      B.lr[off + pos] = B.dL[off + q];
    }
  }
}

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------
#define DC_MERGE()                       \
  const int id = id0 + (int)blockIdx.x;  \
  DcMerge M;                             \
  if (!dc_node(B.n, id, M) || M.N < 2) return;

// Work items: the grid covers the ids id0, id0 + 1, ... of one depth with
// `groups` work-groups each, and a group of 256 threads takes 4 consecutive
// items of its merge, one wave per item.
#define DC_ITEM()                                                   \
  const int id = id0 + (int)(blockIdx.x / (unsigned)groups);        \
  DcMerge M;                                                        \
  if (!dc_node(B.n, id, M) || M.N < 2) return;                      \
  const int lane = threadIdx.x & 63;                                \
  const int item = (int)(blockIdx.x % (unsigned)groups) * 4 +       \
                   __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

__global__ __launch_bounds__(256) void dc_prep(DcBufs B, int id0) {
  DC_MERGE();
  prep_merge(B, id, M);
}
__global__ __launch_bounds__(256) void dc_roots(DcBufs B, int id0, int groups) {
  DC_ITEM();
  root_item(B, id, M, item, lane);
}
__global__ __launch_bounds__(256) void dc_zhat(DcBufs B, int id0, int groups) {
  DC_ITEM();
  zhat_item(B, id, M, item, lane);
}
__global__ __launch_bounds__(256) void dc_rows(DcBufs B, int id0, int groups) {
  DC_ITEM();
  row_item(B, id, M, item, lane);
}
__global__ __launch_bounds__(256) void dc_assemble(DcBufs B, int id0) {
  DC_MERGE();
  assemble_merge(B, id, M);
}

// The five in one launch, a work-group per merge, for depths of small ranges:
// there a launch (4.7 us) costs more than the rounds of roots that each of
// the four waves takes in turn.  Same functions, same results.
__global__ __launch_bounds__(256) void dc_small(DcBufs B, int id0) {
  DC_MERGE();
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  prep_merge(B, id, M);
  __syncthreads();
  for (int i = wave; i < M.N; i += 4) root_item(B, id, M, i, lane);
  __syncthreads();
  if (id != 1) {
    for (int i = wave; i < M.N; i += 4) zhat_item(B, id, M, i, lane);
    __syncthreads();
    for (int i = wave; i < M.N; i += 4) row_item(B, id, M, i, lane);
    __syncthreads();
  }
  assemble_merge(B, id, M);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// Depth of the deepest merge, plus one: the ranges of depth p hold at most
// floor(n / 2^p) entries.
static int dc_depths(int n) {
  int h = 0;
  while ((n >> h) >= 2) ++h;
  return h;
}

void dc_plan(ArenaPlan& p, int n) {
  size_t nn = (size_t)n + 1;
  p.add<double>(nn * 3);          // sig fr lr
  const size_t ids = (size_t)2 << dc_depths(n);  // heap places 0 .. ids - 1
  p.add<double>(2 * ids);         // phi psi
  p.add<double>(nn * 4);          // wd wz wF wL
  p.add<int>(nn);                 // flag
  p.add<double>(nn * 4);          // kd kz kF kL
  p.add<double>(nn * 3);          // dd dF dL
  p.add<int>(nn);                 // org
  p.add<double>(nn * 4);          // tau zh fn ln
  p.add<DcMergeState>(ids / 2);
}

int dc_run(int n, const double* a, const double* b, double* sigma, Arena& ws,
           hipStream_t st) {
  if (n < 1) return DDC_E_ARG;
  const int H = dc_depths(n);  // depths 0 .. H - 1 hold merges, H leaves only
  const size_t ids = (size_t)2 << H;
  size_t nn = (size_t)n + 1;
  DcBufs B;
  B.a = const_cast<double*>(a);
  B.b = const_cast<double*>(b);
  B.sig = ws.take<double>(nn * 3);
  B.fr = B.sig + nn;
  B.lr = B.fr + nn;
  B.phi = ws.take<double>(2 * ids);
  B.psi = B.phi + ids;
  B.wd = ws.take<double>(nn * 4);
  B.wz = B.wd + nn;
  B.wF = B.wz + nn;
  B.wL = B.wF + nn;
  B.flag = ws.take<int>(nn);
  B.kd = ws.take<double>(nn * 4);
  B.kz = B.kd + nn;
  B.kF = B.kz + nn;
  B.kL = B.kF + nn;
  B.dd = ws.take<double>(nn * 3);
  B.dF = B.dd + nn;
  B.dL = B.dF + nn;
  B.org = ws.take<int>(nn);
  B.tau = ws.take<double>(nn * 4);
  B.zh = B.tau + nn;
  B.fn = B.zh + nn;
  B.ln = B.fn + nn;
  B.ms = ws.take<DcMergeState>(ids / 2);
  if (!B.ms) return DDC_E_NOMEM;
  B.n = n;
  B.out = sigma;

  hipLaunchKernelGGL(dc_leaves, dim3((unsigned)ceil_div((int64_t)ids - 1, 256)), dim3(256), 0, st,
                     B, (int)(ids - 1));
  DDC_LAUNCHED();
  if (H == 0) {  // n == 1
    DDC_HIP(hipMemcpyAsync(sigma, B.sig, sizeof(double), hipMemcpyDeviceToDevice, st));
    return DDC_OK;
  }
  for (int p = H - 1; p >= 0; --p) {
    const int id0 = 1 << p;                           // ids id0 .. 2 id0 - 1
    const int groups = (int)ceil_div((int64_t)(n >> p), 4);  // 4 items each
    const unsigned ni = (unsigned)id0 * (unsigned)groups;
    if ((n >> p) <= DC_SMALL) {
      hipLaunchKernelGGL(dc_small, dim3(id0), dim3(256), 0, st, B, id0);
      DDC_LAUNCHED();
      continue;
    }
    hipLaunchKernelGGL(dc_prep, dim3(id0), dim3(256), 0, st, B, id0);
    DDC_LAUNCHED();
    hipLaunchKernelGGL(dc_roots, dim3(ni), dim3(256), 0, st, B, id0, groups);
    DDC_LAUNCHED();
    if (p > 0) {
      hipLaunchKernelGGL(dc_zhat, dim3(ni), dim3(256), 0, st, B, id0, groups);
      DDC_LAUNCHED();
      hipLaunchKernelGGL(dc_rows, dim3(ni), dim3(256), 0, st, B, id0, groups);
      DDC_LAUNCHED();
    }
    hipLaunchKernelGGL(dc_assemble, dim3(id0), dim3(256), 0, st, B, id0);
    DDC_LAUNCHED();
  }
  return DDC_OK;
}

}  // namespace ddc
