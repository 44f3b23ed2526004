// resident.hip -- Golub-Kahan bidiagonalization with the matrix in registers.
//
// Same result as the column steps of bidiag.hip (reference
// bidiag_par.c:34-450: alpha, beta and the unit-norm reflectors in place),
// for matrices, or the last columns of larger ones, that fit the register
// files.  There a column step is bound by latency: bidiag.hip pays two
// kernel launches per step whatever the size (15.6 us per step at 512 x 256,
// 17-20 us up to 2048 x 2048).  Here one launch runs all steps.  The block
// A[k0:m, k0:n] is cut over a grid of work-groups, one per CU, each holding
// its part in registers (512 threads; lane l of a wave holds rows l, l + 64,
// ..., the wave CW columns), and every step updates the part twice (left and
// right reflection) without touching memory.  What the work-groups tell each
// other per step is two short vectors:
//
//   g = A^T c        (c: the current column) sums over the rows: complete in
//                    a wave when one work-group holds all rows (PR = 1), else
//                    summed over the PR = 8 row blocks;
//   h = A r, |r|^2   (r: the current row, after the left update) sums over
//                    the PC column blocks, and the left-updated column k + 1,
//                    from which every work-group forms x = 2 A v and the next
//                    column c.
//
// As in bidiag.hip the products take the raw column and row, and the
// reflectors u = (c + s|c| e)/rl, v = (r + s|r| e)/rl enter afterwards, so
// no exchange is needed for the norms alone.
//
// Per step, three messages follow each other:
//   1 (PR = 8 only) every wave sends its partial g to the eight row blocks'
//     waves that hold the same columns, with row k and |c|^2;
//   2 every work-group sends its partial h, cut into PC segments of rows, to
//     the segments' work-groups, with |r|^2 and column k + 1;
//   3 wave 0 of each work-group forms x and the next c on its segment and
//     publishes them to its row block.
// (Each work-group summing all of h itself, PC R values instead of R + 2 R,
// saves message 3 but reads 16 times as much: 5.7 against 3.4 us per step at
// 512 x 256.)
//
// A message has no flag and there is no barrier over the grid: each word is
// stored once, and its reader polls it until it no longer holds the empty
// mark (the NaN with all bits set, which no arithmetic produces; a NaN to be
// sent is sent in canonical form).  Two things decide the latency:
//  * Words of 1 and 2 go to a box per reader.  A line polled by many waves
//    serves them one after another, and the store that they wait for queues
//    behind them: 13,500 cycles where the 32 work-groups of a row block
//    polled one line of |r|^2, 1,300 with a box each.  Those of 3 have 32
//    readers but each row is read by one wave of each.
//  * The 32 work-groups of a row block share an XCD, so 2 and 3 stay in its
//    L2: a plain store and an sc1 load, 710 cycles one way.  Message 1
//    crosses XCDs by agent-scope stores: 1,770 cycles.
// The row block is the XCD's number as the hardware gives it, the column
// block the work-group's turn on that XCD, so both scopes hold whatever the
// dispatch order.
//
// Emptying.  The reader empties its boxes after it has read them, for use
// two steps later; a producer sends its step e + 2 only after it has read
// this work-group's message of step e + 1, and every wave waits for its
// emptying stores before that message is sent (before the step's first
// barrier, or before its own message 1).  The areas of message 3 are shared:
// in step e each work-group empties its own segment for step e + 2, last
// used in step e - 2 (a ring of four).  By then it has read every segment of
// step e, whose senders had all their waves through step e - 2.
//
// Per step at 2048 x 1024, in cycles of wave 0 (stamped build, 11,400 in all,
// 4.6 us): products 470, message 1 3,700, reflector and left update 840, sum
// over waves and barrier 1,400, sending 670, message 2 1,350, x 850, message
// 3 and barrier 1,550, right update 540.  By kernel trace, per step: 1.9 us
// (128 x 64, one work-group), 2.8 (256 x 256), 3.4 (512 x 256), 4.35 (1024^2),
// 5.9 (2048^2), 8.2 (3072^2), where bidiag.hip takes 14-20 us.  Sums in a
// fixed order: results are bitwise reproducible.
//
// The polls need every work-group of the grid to be resident at once.  Each
// launch starts with a rendezvous (bounded wait): if the work-groups do not
// all arrive, because other work holds the CUs, the kernel ends without
// having changed anything and the caller runs the steps by bidiag.hip.
// After it no wait can fail; the polls are bounded all the same.
#include <algorithm>

#include "ddc_common.h"
#include "householder.h"

namespace ddc {

namespace {

constexpr int RS_T = 512;             // threads per work-group (256 registers each)
constexpr int RS_W = RS_T / 64;       // waves
constexpr int RS_RING = 2;            // steps the boxes hold
constexpr int RS_XRING = 4;           // steps the areas of x hold
constexpr int RS_LAUNCH = 15;         // launches of one bidiagonalization at most
constexpr int RS_SYNC = 16 * RS_LAUNCH + 1;  // sync words
// The rendezvous' wait in polls: 0.9 ms, with the work-groups of one XCD or of all.
// Those of a free GPU start within some tens of microseconds; where other work
// holds its CUs, those that wait hold CUs themselves, so what is lost to both is
// kept small beside the panel kernels' time (100,000 polls lasted 30 ms in a call
// of 3.1 ms).  A bound by the clock, read in this loop, cost every launch 4 us.
constexpr int RS_RDV = 3000;
constexpr int RS_POLLS = 1 << 21;     // polls of one exchange before it is given up
// before the first poll of message 1, in units of 64 cycles: it cannot have
// come sooner (polls in flight delay it: two of them staggered by half a
// round trip cost 800 cycles per step)
constexpr int RS_G_SLEEP = 8;
constexpr double RS_SWITCH_US = 30.0;  // cost of going on in another launch
typedef unsigned long long u64;
constexpr u64 RS_EMPTY = ~0ull;
constexpr u64 RS_NAN = 0x7ff8000000000000ull;

// s_getreg operand: bits 0-3 of register 20, XCC_ID (the number of the XCD)
constexpr int RS_XCC_ID = 20 | (3 << 11);

// sync words of launch i from 16 i: arrivals, state, turns by XCD; RS_STATUS:
// 0, 1 + i (launch i did not assemble), RS_FAILED (an exchange gave up)
constexpr int RS_STATUS = RS_SYNC - 1;
constexpr unsigned RS_GO = 1, RS_STOP = 2, RS_FAILED = 1000;

template <typename TS>
struct ResArgs {
  int m, n, lda, k0, k1, idx;
  unsigned groups;  // work-groups that the launch waits for
  TS* A;
  double* alpha;
  double* beta;
  u64* gx;  // boxes of g: [slot][b][p][wave][g_box]
  u64* hx;  // boxes of h: [slot][b][p][h_box]
  u64* xx;  // areas of x: [slot][b][x_area]
  unsigned* sync;
};

__device__ __forceinline__ void put(u64* p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void put(u64* p, double v) {
  put(p, v == v ? __builtin_bit_cast(u64, v) : RS_NAN);
}
__device__ __forceinline__ u64 take(const u64* p) {
  return __hip_atomic_load(const_cast<u64*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The same through a buffer resource: word soff (wave-uniform) + voff of it.
// (Aux bit 4: sc1, the agent scope; an 8-byte load is a single access.  The
// caller's loop holds a compiler barrier, so that every poll loads anew.)
__device__ __forceinline__ u64 take(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return __builtin_bit_cast(u64, __builtin_amdgcn_raw_buffer_load_b64(r, voff * 8, soff * 8, 16));
}
// Between work-groups of one XCD: a plain store (through the write-through L1)
// stays in the XCD's L2, where the sc1 loads of its other work-groups find
// it: 710 cycles one way, against 1590 with the agent-scope store, which goes
// on to memory, and 1770 to another XCD (where plain stores are not seen).
__device__ __forceinline__ void put_l2(u64* p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void put_l2(u64* p, double v) {
  put_l2(p, v == v ? __builtin_bit_cast(u64, v) : RS_NAN);
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t ring_rsrc(const u64* p, int64_t words) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<u64*>(p), 0, (int)(words * 8), 0x00020000);
}
__device__ __forceinline__ unsigned take(const unsigned* p) {
  return __hip_atomic_load(const_cast<unsigned*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double val(u64 v) { return __builtin_bit_cast(double, v); }
// the stores of this wave have reached the agent's coherence point (in the
// place it is called, after polls, nothing is left to wait for)
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

constexpr int pow2_ceil(int x) {
  int p = 1;
  while (p < x) p *= 2;
  return p;
}
// words of a box of g (one per receiving row block, column block and wave):
// the eight partials of the CW sums, of |c|^2, row k on the CW columns and
// its entry of c
constexpr int g_box(int CW) { return (9 * CW + 9 + 15) / 16 * 16; }
// words of a box of h (one per work-group): the PC partials of its segment of
// SEG rows (R in all), column k + 1 there, |r|^2 by column block and r_{k+1}
constexpr int h_box(int R, int PC) { return R + (R / PC + 15) / 16 * 16 + 64; }
// words of x, one area per row block: x and the next column on R rows
constexpr int x_area(int R) { return 2 * R; }

// What a reflection needs of Refl: s|x|, rl and 1/rl.  |x| and 1/rl by
// Goldschmidt and Newton steps from the hardware's reciprocal square root
// (within an ulp or two): each of these scalars is on the serial chain of a
// column step, and the library's square roots and division took 0.16 us of
// it, twice per step.  Sums of squares near the ends of the range, zero
// among them, go through Refl.
struct Scal {
  double diag, sn, rl, ir;
  __device__ __forceinline__ void make(double ss, double x1) {
    if (ss >= 0x1p-900 && ss <= 0x1p900) {
      const double y = __builtin_amdgcn_rsq(ss);
      double g = ss * y, h = 0.5 * y;
      const double e = fma(-h, g, 0.5);
      g = fma(g, e, g);
      h = fma(h, e, h);
      const double nrm = fma(fma(-g, g, ss), h, g);
      const double t = 2.0 * nrm * (nrm + fabs(x1));  // rl^2
      const double z = __builtin_amdgcn_rsq(t);
      const double f = fma(-t * z, z, 1.0);
      ir = fma(z * f, fma(0.375, f, 0.5), z);
      rl = t * ir;
      sn = x1 < 0 ? -nrm : nrm;
      diag = -sn;
    } else {
      Refl R;
      R.make(ss, x1);
      sn = R.sgn * R.nrm;
      rl = R.rl;
      ir = rl != 0.0 ? 1.0 / rl : 0.0;
      diag = R.diag();
    }
  }
  __device__ __forceinline__ void none() { rl = ir = 0.0; }
};

}  // namespace

// RL: rows per lane, CW: columns per wave, PR: row blocks (1 or 8), PC:
// column blocks.  The block at k0 must have at most 64 RL PR rows and 8 CW PC
// columns.  Column k0 + j lives in column block j % PC, wave (j / PC) % 8.
template <typename TS, int RL, int CW, int PR, int PC>
__global__ __launch_bounds__(RS_T, 1) void bd_resident(ResArgs<TS> g) {
  static_assert(PR == 1 || (PR == 8 && PC == 32), "grid shapes of the exchanges");
  constexpr int R = 64 * RL, RW = R / RS_W;  // rows per work-group, per wave's segment
  constexpr int NV = pow2_ceil(CW), LGD = 64 / NV;  // wave_scatter's groups
  constexpr int LG = PR > 1 ? 8 : LGD;              // lanes per column after the sums
  constexpr int NG = PR > 1 ? (CW + 7) / 8 : 1;     // column groups of a wave
  static_assert(NV <= 16, "wave_scatter takes up to 16 values");
  constexpr int NCH = (RW + 63) / 64;  // 64-row chunks of a wave's segment
  // rows a work-group reduces, and how a wave's lanes take them: SEGP rows by
  // PP partials side by side, NPL reads
  constexpr int SEG = R / PC, SEGP = SEG < 64 ? pow2_ceil(SEG) : 64;
  constexpr int PP = 64 / SEGP, NPL = PC > PP ? PC / PP : 1;
  static_assert(PC == 1 || (SEG <= 64 && PC % PP == 0), "one wave reads a segment");
  __shared__ double hp[RS_W][R];       // h by wave
  __shared__ double xs[R], cs[R];  // x and the next column
  __shared__ double rowk[RS_W][CW + 1];  // row k on the wave's columns, c_k
  __shared__ double rrp[RS_W];
  __shared__ double sv[5];  // right reflection: sn, rl, 1/rl, diag, r_{k+1}
  __shared__ double colb[PC == 1 ? R : 1], rk1b;
  __shared__ double vst[RS_W][CW];  // the last step's right reflector on the wave's columns
  __shared__ int s_go, s_dead;

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  int b = 0, p = 0;
  if constexpr (PR * PC > 1) {
    // the row block is the XCD's number, the column block the work-group's
    // turn on that XCD (one more than its CUs take never gets one)
    const int xcc = __builtin_amdgcn_s_getreg(RS_XCC_ID);
    if (PR == 1 && xcc != 0) return;  // one XCD's work-groups
    if (tid == 0) s_go = xcc < 8 ? (int)atomicAdd(g.sync + 16 * g.idx + 2 + (xcc & 7), 1u) : PC;
    __syncthreads();
    p = __builtin_amdgcn_readfirstlane(s_go);
    if (p >= PC) return;
    b = PR > 1 ? xcc : 0;
  }
  const int m = g.m, n = g.n, lda = g.lda, k0 = g.k0;
  const int row0 = k0 + b * R;  // global row of local row 0

  // column k0 on this lane's rows, before the rendezvous: after it, its owner
  // may overwrite it with the reflector
  double c[RL];
#pragma unroll
  for (int q = 0; q < RL; ++q) {
    const int r = row0 + 64 * q + lane;
    c[q] = r < m ? (double)g.A[r + (int64_t)k0 * lda] : 0.0;
  }
  // (loaded, not only issued)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  // rendezvous
  if (tid == 0) {
    s_dead = 0;
    bool go = take(g.sync + RS_STATUS) == 0;
    if constexpr (PR * PC > 1) {
      unsigned* arrived = g.sync + 16 * g.idx;
      unsigned* state = arrived + 1;
      if (go) {
        if (atomicAdd(arrived, 1u) + 1 == g.groups) atomicCAS(state, 0u, RS_GO);
        for (int i = 0; i < RS_RDV && take(state) == 0; ++i) __builtin_amdgcn_s_sleep(8);
        // all decide alike: whoever writes the state first decides
        atomicCAS(state, 0u, RS_STOP);
        go = take(state) == RS_GO;
        if (!go) atomicCAS(g.sync + RS_STATUS, 0u, 1u + (unsigned)g.idx);
      }
    }
    s_go = go;
  }
  __syncthreads();
  if (!s_go) return;

  double a[RL][CW];
#pragma unroll
  for (int s = 0; s < CW; ++s) {
    const int j = k0 + p + PC * (w + RS_W * s);
#pragma unroll
    for (int q = 0; q < RL; ++q) {
      const int r = row0 + 64 * q + lane;
      a[q][s] = (j < n && r < m) ? (double)g.A[r + (int64_t)j * lda] : 0.0;
    }
  }
  const int sg = lane / LG;  // this lane's column of the wave (of group 0)
  constexpr int64_t GBOX = g_box(CW), GSLOT = PR * PC * RS_W * GBOX;
  constexpr int64_t HBOX = h_box(R, PC), HSLOT = PR * PC * HBOX;
  // parts of a box of h
  constexpr int BC = R, BS = BC + (SEG + 15) / 16 * 16;
  constexpr int64_t XSLOT = PR * x_area(R);  // parts: x, next column from R
  u64* const xarea = PC > 1 ? g.xx + (int64_t)b * x_area(R) : nullptr;
  // this wave's box of g, this work-group's box of h (slot 0)
  u64* const gbox = PR > 1 ? g.gx + ((int64_t)(b * PC + p) * RS_W + w) * GBOX : nullptr;
  u64* const hbox = PC > 1 ? g.hx + (int64_t)(b * PC + p) * HBOX : nullptr;
  // where it sends: row block j's box of g, column block j's box of h
  u64* const gout = PR > 1 ? g.gx + (int64_t)(p * RS_W + w) * GBOX : nullptr;
  constexpr int64_t GSTEP = PC * RS_W * GBOX;
  u64* const hout = PC > 1 ? g.hx + (int64_t)b * PC * HBOX : nullptr;
  const __amdgpu_buffer_rsrc_t grs = ring_rsrc(gbox, PR > 1 ? (RS_RING - 1) * GSLOT + GBOX : 0);
  const __amdgpu_buffer_rsrc_t hrs = ring_rsrc(hbox, PC > 1 ? (RS_RING - 1) * HSLOT + HBOX : 0);
  const __amdgpu_buffer_rsrc_t xrs =
      ring_rsrc(xarea, PC > 1 ? (RS_XRING - 1) * XSLOT + x_area(R) : 0);
  bool dead = false;
  // polls of one exchange: true to go on polling
  auto again = [&](bool empty, int& tries) {
    if (!__any(empty)) return false;
    ++tries;
    if (tries < RS_POLLS &&
        ((tries & 1023) != 0 || take(g.sync + RS_STATUS) != RS_FAILED))
      return true;
    dead = true;  // and everyone else with it
    if (lane == 0)
      __hip_atomic_store(g.sync + RS_STATUS, RS_FAILED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return false;
  };

  // the reflectors, stored by their columns' owners (u, of column k0 + kk, held
  // in c) and, of the rows' entries, by each column's (v, of row k0 + kk, in LDS)
  // (the empty asm keeps addresses and masks from being held in registers
  // through all steps)
  auto store_u = [&](int kk) {
    if (p == kk % PC && w == (kk / PC) % RS_W) {
      int r = row0 + lane;
      asm volatile("" : "+v"(r));
      TS* const col = g.A + (int64_t)(k0 + kk) * lda;
#pragma unroll
      for (int q = 0; q < RL; ++q)
        if (r + 64 * q >= k0 + kk && r + 64 * q < m) col[r + 64 * q] = (TS)c[q];
    }
  };
  auto store_v = [&](int kk) {
    if (kk >= 0 && b == kk % PR && lane < CW) {
      const int jj = p + PC * (w + RS_W * lane);
      if (jj > kk && k0 + jj < n) g.A[k0 + kk + (int64_t)(k0 + jj) * lda] = (TS)vst[w][lane];
    }
  };
  int vrow = -1;  // the step whose v is still to be stored
  for (int kk = 0; k0 + kk < g.k1; ++kk) {
    const int k = k0 + kk;
    const bool last_row = m < n && k == m - 1;  // wide: no left reflection
    const int slot = kk % RS_RING;
    const int kr = k - row0;  // row k in this row block (outside: not held)
    const bool own_k = kr >= 0 && kr < R;

    // ---- g = A^T c, row k and |c|^2 ----
    double gl[NG], ak[NG], ck, cn = 0.0;  // cn: |c|^2, here over this row block
    {
#pragma unroll
      for (int q = 0; q < RL; ++q) cn += c[q] * c[q];
      cn = wave_total(cn);
      double d[NV];
#pragma unroll
      for (int s = 0; s < NV; ++s) {
        d[s] = 0.0;
        if (s < CW) {
#pragma unroll
          for (int q = 0; q < RL; ++q) d[s] += a[q][s < CW ? s : 0] * c[q];
        }
      }
      const double dl = wave_scatter<NV>(d);
      if (own_k) {
#pragma unroll
        for (int q = 0; q < RL; ++q)
          if (q == kr >> 6 && lane == (kr & 63)) {
#pragma unroll
            for (int s = 0; s < CW; ++s) rowk[w][s] = a[q][s];
            rowk[w][CW] = c[q];
          }
        wave_fence();
      }
      if constexpr (PR == 1) {
        gl[0] = dl;
        ak[0] = rowk[w][min(sg, CW - 1)];
        ck = rowk[w][CW];
      } else {
        u64* const gs = gout + slot * GSLOT;
        const int sd = lane / LGD;
        stores_done();
#pragma unroll
        for (int j = lane % LGD; j < PR; j += LGD)
          if (sd < CW) put(gs + j * GSTEP + 8 * sd + b, dl);
        if (lane < PR) put(gs + lane * GSTEP + 8 * CW + b, cn);
        if (own_k)
          for (int i = lane; i < PR * (CW + 1); i += 64)
            put(gs + i / (CW + 1) * GSTEP + 8 * CW + 8 + i % (CW + 1), rowk[w][i % (CW + 1)]);
        u64 vg[NG], va[NG], vn, vc;
        int tries = 0;
        bool empty;
        const int so = (int)(slot * GSLOT);
        __builtin_amdgcn_s_sleep(RS_G_SLEEP);
        do {
          asm volatile("" ::: "memory");
          empty = false;
#pragma unroll
          for (int i = 0; i < NG; ++i) {
            const int s = min(sg + 8 * i, CW - 1);
            vg[i] = take(grs, 8 * s + (lane & 7), so);
            va[i] = take(grs, 8 * CW + 8 + s, so);
            empty |= vg[i] == RS_EMPTY || va[i] == RS_EMPTY;
          }
          vn = take(grs, 8 * CW + (lane & 7), so);
          vc = take(grs, 9 * CW + 8, so);
          empty |= vn == RS_EMPTY || vc == RS_EMPTY;
        } while (again(empty, tries));
        u64* const ge = gbox + slot * GSLOT;
        for (int i = lane; i < 9 * CW + 9; i += 64) put(ge + i, RS_EMPTY);
        auto sum8 = [](double v) {
          v += dpp_all<DPP_XOR1>(v);
          v += dpp_all<DPP_XOR2>(v);
          return v + dpp_all<DPP_HALF_MIRROR>(v);
        };
#pragma unroll
        for (int i = 0; i < NG; ++i) {
          gl[i] = sum8(val(vg[i]));
          ak[i] = val(va[i]);
        }
        cn = sum8(val(vn));
        ck = val(vc);
      }
    }

    // ---- left reflector; y = 2 A^T u and row k on this lane's columns ----
    Scal L;
    L.make(cn, ck);
    if (last_row) L.none();
    const double uk = rl_quot(ck + L.sn, L.rl, L.ir);
    double yl[NG], rr[NG];
#pragma unroll
    for (int i = 0; i < NG; ++i) {
      const int s = sg + 8 * i;
      const int jj = p + PC * (w + RS_W * s);
      const bool live = s < CW && jj > kk && k0 + jj < n;
      yl[i] = live ? 2.0 * rl_quot(gl[i] + L.sn * ak[i], L.rl, L.ir) : 0.0;
      rr[i] = live ? ak[i] - uk * yl[i] : 0.0;
    }
    double h[RL], r2 = 0.0;
#pragma unroll
    for (int q = 0; q < RL; ++q) {
      // from here on c[q] holds the reflector's entry
      c[q] = rl_quot(64 * q + lane == kr ? c[q] + L.sn : c[q], L.rl, L.ir);
      h[q] = 0.0;
    }
    if (b == 0 && p == 0 && tid == 0) g.alpha[k] = last_row ? ck : L.diag;
#pragma unroll
    for (int s = 0; s < CW; ++s) {
      const double ys = lane_value(yl[s / 8 * (NG > 1)], NG > 1 ? (s & 7) * LG : s * LG);
      const double rs = lane_value(rr[s / 8 * (NG > 1)], NG > 1 ? (s & 7) * LG : s * LG);
      r2 += rs * rs;
#pragma unroll
      for (int q = 0; q < RL; ++q) {
        a[q][s] -= c[q] * ys;
        h[q] += a[q][s] * rs;
      }
    }

    // ---- h = A r over the work-group's columns, column k + 1 ----
#pragma unroll
    for (int q = 0; q < RL; ++q) hp[w][64 * q + lane] = h[q];
    if (lane == 0) {
      rrp[w] = r2;
      if (dead) s_dead = 1;
    }
    u64* const hs = PC > 1 ? hout + slot * HSLOT : nullptr;
    // local column k + 1; in the last step of m >= n, a left reflection only
    // (r = 0, so no right one follows), any column
    const int j1 = min(kk + 1, PC * RS_W * CW - 1);
    if (p == j1 % PC && w == (j1 / PC) % RS_W) {
      const int s1 = j1 / (PC * RS_W);
#pragma unroll
      for (int s = 0; s < CW; ++s)
        if (s == s1) {
#pragma unroll
          for (int q = 0; q < RL; ++q) {
            if constexpr (PC > 1)
              put_l2(hs + (64 * q + lane) / SEG * HBOX + BC + (64 * q + lane) % SEG, a[q][s]);
            else colb[64 * q + lane] = a[q][s];
          }
          const double rk1 = lane_value(rr[s / 8 * (NG > 1)], NG > 1 ? (s & 7) * LG : s * LG);
          if constexpr (PC > 1) {
            if (lane < PC) put_l2(hs + lane * HBOX + BS + PC, rk1);
          } else if (lane == 0) {
            rk1b = rk1;
          }
        }
    }
    stores_done();  // the emptying of this wave's boxes: long since
    __syncthreads();
    if (s_dead) break;
    const bool noright = k == n - 2 && !last_row;  // one entry left: beta as it stands
    Scal V;
    double x[RL], rk1;
    // x = 2 A v and the next column on one row, from h, column k + 1 and v_{k+1}
    auto finish = [&](double h, double col, double v1, bool in, double& x, double& cx) {
      x = in ? 2.0 * rl_quot(h + V.sn * col, V.rl, V.ir) : 0.0;
      cx = in ? col - x * v1 : 0.0;
    };
    if constexpr (PC > 1) {
      for (int r = tid; r < R; r += RS_T) {
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < RS_W; ++i) s += hp[i][r];
        put_l2(hs + r / SEG * HBOX + p * SEG + r % SEG, s);
      }
      if (w == 1 && lane < PC) {
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < RS_W; ++i) s += rrp[i];
        put_l2(hs + lane * HBOX + BS + p, s);
      }
      // (stores whose completion nothing waits for soon: before the sending,
      // their acknowledgements would delay it)
      store_u(kk);
      store_v(vrow);
      const int so = (int)(slot * HSLOT), xo = (int)(kk % RS_XRING * XSLOT);
      u64* const xs_out = xarea + xo;
      bool empty;
      int tries = 0;
      if (w == 0) {
        // wave 0: the right reflection and this work-group's segment
        const int sl = min(lane % SEGP, SEG - 1);
        u64 vr, vh[NPL], vc;
        do {
          asm volatile("" ::: "memory");
          vr = take(hrs, BS + min(lane, PC), so);
          vc = take(hrs, BC + sl, so);
          empty = vr == RS_EMPTY || vc == RS_EMPTY;
#pragma unroll
          for (int i = 0; i < NPL; ++i) {
            vh[i] = take(hrs, lane / SEGP * SEG + sl, so + i * PP * SEG);
            empty |= vh[i] == RS_EMPTY;
          }
        } while (again(empty, tries));
        rk1 = lane_value(val(vr), PC);
        V.make(wave_total(lane < PC ? val(vr) : 0.0), rk1);
        if (noright) V.none();
        double h = 0.0;
#pragma unroll
        for (int i = 0; i < NPL; ++i) h += val(vh[i]);
        if constexpr (PP >= 2) h = half_sum<32>(h);
        if constexpr (PP >= 4) h = half_sum<16>(h);
        if constexpr (PP >= 8) h += dpp_all<DPP_ROR8>(h);
        if constexpr (PP >= 16) h += dpp_all<DPP_ROR4>(h);
        double xl, cl;
        finish(h, val(vc), rl_quot(rk1 + V.sn, V.rl, V.ir), p * SEG + sl > kr, xl, cl);
        if (lane < SEG) {
          put_l2(xs_out + p * SEG + lane, xl);
          put_l2(xs_out + R + p * SEG + lane, cl);
        }
        if (lane == 0) {
          sv[0] = V.sn;
          sv[1] = V.rl;
          sv[2] = V.ir;
          sv[3] = V.diag;
          sv[4] = rk1;
        }
      }
      // every wave: its share of the rows of x and the next column
      u64 vx[NCH], vn[NCH];
      tries = 0;
      do {
        asm volatile("" ::: "memory");
        empty = false;
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
          const int row = w * RW + min(64 * i + lane, RW - 1);
          vx[i] = take(xrs, row, xo);
          vn[i] = take(xrs, R + row, xo);
          empty |= vx[i] == RS_EMPTY || vn[i] == RS_EMPTY;
        }
      } while (again(empty, tries));
#pragma unroll
      for (int i = 0; i < NCH; ++i)
        if (64 * i + lane < RW) {
          const int row = w * RW + 64 * i + lane;
          xs[row] = val(vx[i]);
          cs[row] = val(vn[i]);
        }
    } else {
      store_u(kk);
      store_v(vrow);
      rk1 = rk1b;
      double rn = 0.0;
#pragma unroll
      for (int i = 0; i < RS_W; ++i) rn += rrp[i];
      V.make(rn, rk1);
      if (noright) V.none();
      const double v1 = rl_quot(rk1 + V.sn, V.rl, V.ir);
#pragma unroll
      for (int ch = 0; ch < NCH; ++ch) {
        const int rl = ch * 64 + lane, row = w * RW + min(rl, RW - 1);
        double h = 0.0, xl, cl;
#pragma unroll
        for (int i = 0; i < RS_W; ++i) h += hp[i][row];
        finish(h, colb[row], v1, rl < RW && row > kr, xl, cl);
        if (rl < RW) {
          xs[row] = xl;
          cs[row] = cl;
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < RL; ++q) x[q] = xs[64 * q + lane];
    if constexpr (PC > 1) {
      // the box for step e + 2, and this work-group's part of the area of x
      // for the same step (used in step e - 2)
      u64* const box = hbox + slot * HSLOT;
      u64* const xe = xarea + (kk + 2) % RS_XRING * XSLOT;
      for (int r = tid; r < R; r += RS_T) put_l2(box + r, RS_EMPTY);
      if (w == 2 && lane < SEG) put_l2(box + BC + lane, RS_EMPTY);
      if (w == 3 && lane <= PC) put_l2(box + BS + lane, RS_EMPTY);
      if (w == 4 && lane < SEG) put_l2(xe + p * SEG + lane, RS_EMPTY);
      if (w == 5 && lane < SEG) put_l2(xe + R + p * SEG + lane, RS_EMPTY);
      V.sn = sv[0];
      V.rl = sv[1];
      V.ir = sv[2];
      V.diag = sv[3];
      rk1 = sv[4];
    }
    // ---- right update ----
    vrow = kk;
    double vl[NG];
#pragma unroll
    for (int i = 0; i < NG; ++i) {
      const int s = sg + 8 * i;
      const int jj = p + PC * (w + RS_W * s);
      const bool live = s < CW && jj > kk && k0 + jj < n;
      vl[i] = live ? rl_quot(jj == j1 ? rr[i] + V.sn : rr[i], V.rl, V.ir) : 0.0;
      if (s < CW && lane % LG == 0) vst[w][s] = vl[i];
    }
    if (b == 0 && p == 0 && tid == 0 && k < n - 1) g.beta[k] = noright ? rk1 : V.diag;
#pragma unroll
    for (int s = 0; s < CW; ++s) {
      const double vs = lane_value(vl[s / 8 * (NG > 1)], NG > 1 ? (s & 7) * LG : s * LG);
#pragma unroll
      for (int q = 0; q < RL; ++q) a[q][s] -= x[q] * vs;
    }
#pragma unroll
    for (int q = 0; q < RL; ++q) c[q] = cs[64 * q + lane];
  }

  store_v(vrow);
  // what is left for the next launch
  if (g.k1 < min(m, n)) {
    // (addresses formed anew: kept from the loads at the start they would
    // take two registers per entry through all steps)
    int r0 = row0 + lane, j0 = k0 + p + PC * w;
    asm volatile("" : "+v"(r0), "+v"(j0));
#pragma unroll
    for (int s = 0; s < CW; ++s) {
      const int j = j0 + PC * RS_W * s;
#pragma unroll
      for (int q = 0; q < RL; ++q) {
        const int r = r0 + 64 * q;
        if (j >= g.k1 && j < n && r >= g.k1 && r < m) g.A[r + (int64_t)j * lda] = (TS)a[q][s];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

namespace {

// A kernel shape: at most 64 RL PR rows and 8 CW PC columns.  step_us: time
// of a column step, as measured by kernel trace (launch time over its steps).
template <typename TS>
struct ResShape {
  int rl, cw, pr, pc;
  double step_us;
  void (*kern)(ResArgs<TS>);
  int rows() const { return 64 * rl * pr; }
  int cols() const { return RS_W * cw * pc; }
};
#define RS_SHAPE(RL, CW, PR, PC, US) {RL, CW, PR, PC, US, &bd_resident<TS, RL, CW, PR, PC>}
template <typename TS>
const ResShape<TS>* res_shapes(int* count) {
  // by falling time per step
  static const ResShape<TS> tab[] = {
      RS_SHAPE(16, 4, 8, 32, 10.5), RS_SHAPE(6, 12, 8, 32, 8.2), RS_SHAPE(8, 8, 8, 32, 6.7),
      RS_SHAPE(16, 2, 8, 32, 6.1),  RS_SHAPE(4, 8, 8, 32, 5.9),  RS_SHAPE(8, 4, 8, 32, 5.3),
      RS_SHAPE(4, 4, 8, 32, 4.65),  RS_SHAPE(8, 2, 8, 32, 4.55), RS_SHAPE(2, 4, 8, 32, 4.35),
      RS_SHAPE(4, 2, 8, 32, 4.0),   RS_SHAPE(2, 2, 8, 32, 3.8),  RS_SHAPE(8, 2, 1, 32, 3.5),
      RS_SHAPE(8, 1, 1, 32, 3.4),   RS_SHAPE(4, 1, 1, 32, 2.8),  RS_SHAPE(2, 16, 1, 1, 2.7),
      RS_SHAPE(2, 8, 1, 1, 1.9),
  };
  *count = (int)(sizeof(tab) / sizeof(tab[0]));
  return tab;
}
#undef RS_SHAPE

// The last shape (fastest step) that holds rows x cols, or -1.
template <typename TS>
int res_pick(int rows, int cols) {
  int cnt;
  const ResShape<TS>* t = res_shapes<TS>(&cnt);
  for (int i = cnt - 1; i >= 0; --i)
    if (t[i].rows() >= rows && t[i].cols() >= cols) return i;
  return -1;
}

template <typename TS>
int64_t res_g_words(const ResShape<TS>& s) {
  return s.pr > 1 ? (int64_t)RS_RING * s.pr * s.pc * RS_W * g_box(s.cw) : 0;
}
template <typename TS>
int64_t res_h_words(const ResShape<TS>& s) {
  return s.pc > 1 ? (int64_t)RS_RING * s.pr * s.pc * h_box(64 * s.rl, s.pc) : 0;
}
template <typename TS>
int64_t res_words(const ResShape<TS>& s) {
  return res_g_words(s) + res_h_words(s) +
         (s.pc > 1 ? (int64_t)RS_XRING * s.pr * x_area(64 * s.rl) : 0);
}

}  // namespace

// Whether the current device has the 256 CUs the grids assume.
static bool res_device() {
  static int cus[64];  // by device: 0 not asked yet
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return false;
  if (cus[dev] == 0 &&
      hipDeviceGetAttribute(&cus[dev], hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
    (void)hipGetLastError();
    cus[dev] = -1;
  }
  return cus[dev] >= 256;
}

// First column step from which the resident kernels can run an m x n
// bidiagonalization, on a multiple of `align`, or -1.
template <typename TS>
int resident_first(int m, int n, int align) {
  if (!res_device()) return -1;
  const int mn = std::min(m, n);
  for (int k = 0; k < mn; k += align)
    if (res_pick<TS>(m - k, n - k) >= 0) return k;
  return -1;
}

void resident_plan(ArenaPlan& p) {
  int cnt;
  const ResShape<double>* t = res_shapes<double>(&cnt);
  int64_t mx = 0;
  for (int i = 0; i < cnt; ++i) mx = std::max(mx, res_words(t[i]));
  p.add<u64>((size_t)mx);
  p.add<unsigned>(RS_SYNC);
}

__global__ __launch_bounds__(1024) void rs_clear(unsigned* sync, double* beta, int nb) {
  for (int i = threadIdx.x; i < RS_SYNC; i += 1024) sync[i] = 0;
  for (int i = threadIdx.x; i < nb; i += 1024) beta[i] = 0.0;
}

// Column steps k0 .. min(m, n) - 1 of the bidiagonalization of A, whose
// block A[k0:m, k0:n] must be fully updated.  *done: the steps completed
// (less than min(m, n) if a launch did not assemble; A is then fully updated
// from *done, a multiple of align, on).
template <typename TS>
int resident_run(int m, int n, TS* A, int lda, double* alpha, double* beta, int k0, int align,
                 Arena& ws, hipStream_t st, int* done, int absent) {
  int cnt;
  const ResShape<TS>* tab = res_shapes<TS>(&cnt);
  int64_t mx = 0;
  for (int i = 0; i < cnt; ++i) mx = std::max(mx, res_words(tab[i]));
  u64* ring = ws.take<u64>((size_t)mx);
  unsigned* sync = ws.take<unsigned>(RS_SYNC);
  if (!sync) return DDC_E_NOMEM;
  // beta too where nothing before this call has cleared it
  hipLaunchKernelGGL(rs_clear, dim3(1), dim3(1024), 0, st, sync, beta, k0 == 0 ? n : 0);
  DDC_LAUNCHED();
  const int mn = std::min(m, n);
  int start[RS_LAUNCH];  // first step of each launch
  int nl = 0;
  *done = k0;
  for (int k = k0; k < mn;) {
    const int i = res_pick<TS>(m - k, n - k);
    if (i < 0 || nl == RS_LAUNCH) return DDC_E_ARG;
    const ResShape<TS>& s = tab[i];
    // up to where a faster shape holds the rest for long enough to pay for
    // another launch
    int k1 = mn;
    for (int f = cnt - 1; f > i; --f) {
      const int kf = (int)round_up(std::max({k + 1, m - tab[f].rows(), n - tab[f].cols()}), align);
      if (kf < k1 && (mn - kf) * (s.step_us - tab[f].step_us) > RS_SWITCH_US) k1 = kf;
    }
    ResArgs<TS> a;
    a.m = m;
    a.n = n;
    a.lda = lda;
    a.k0 = k;
    a.k1 = k1;
    a.idx = nl;
    a.groups = (unsigned)(s.pr * s.pc) + (nl == absent ? 1u : 0u);
    a.A = A;
    a.alpha = alpha;
    a.beta = beta;
    a.gx = ring;
    a.hx = ring + res_g_words(s);
    a.xx = a.hx + res_h_words(s);
    a.sync = sync;
    if (res_words(s) > 0)
      DDC_HIP(hipMemsetAsync(ring, 0xff, sizeof(u64) * (size_t)res_words(s), st));
    const int grid = s.pr > 1 ? s.pr * s.pc : (s.pc > 1 ? 8 * s.pc : 1);
    hipLaunchKernelGGL(s.kern, dim3(grid), dim3(RS_T), 0, st, a);
    DDC_LAUNCHED();
    start[nl++] = k;
    k = k1;
  }
  unsigned status = 0;
  DDC_TRY(host_read(&status, sync + RS_STATUS, sizeof(status), st));
  if (status == RS_FAILED) {
    report_error("an exchange of the bidiagonalization's work-groups gave up");
    return DDC_E_HIP;
  }
  *done = status == 0 ? mn : start[status - 1];
  return DDC_OK;
}

template int resident_first<double>(int, int, int);
template int resident_first<float>(int, int, int);
template int resident_run<double>(int, int, double*, int, double*, double*, int, int, Arena&,
                                  hipStream_t, int*, int);
template int resident_run<float>(int, int, float*, int, double*, double*, int, int, Arena&,
                                 hipStream_t, int*, int);

}  // namespace ddc
