// bjlines.hip -- line-wavefront form of the block-Jacobi apply, FP64 and
// double-double.
//
// A block is a run of consecutive rows of a natural-order grid (lines of nx
// cells, planes of whole lines) whose factor rows couple only to the cell
// neighbour (offset 1), the line neighbour (offset nx) and the plane neighbour
// (offset nxy).  The block is cut into pieces, one per plane it touches, and
// a piece into groups of 64 lines, one wavefront each.  In sweep coordinates
// (backward: cells, lines and planes counted from the other end) lane l of a
// wavefront computes cell c of its line at step t = c + tw + l, where
//   tw = 64 jw + 8 jw + 9 k   (line group jw of piece k; 9 k only where the
//                              block couples planes)
// so that the cell neighbour was computed by the thread itself at step t - 1,
// the line neighbour by the lane below at t - 1 (a DPP wave shift) or, for
// lane 0, by lane 63 of the wavefront before at t - 9, and the plane
// neighbour by the same lane of the plane's wavefront at t - 9.  Values older
// than a step come from a ring of the last 24 steps of every line in LDS; one
// LDS barrier per group of kLG = 8 steps publishes them (a value of step t - 9
// or earlier belongs to an earlier group).  A block may begin and end inside
// a line or a plane: cells of its lines outside its rows are swept as if the
// lines were whole, their value replaced by the one an absent neighbour has.
// Every row sums its couplings in the stored order with the same operations
// as the level-scheduled kernels, so the values are bit-identical to theirs.
//
// What bounds it: with few blocks (64 on 256 CUs) the sweep is one dependent
// chain of steps and a lone wavefront per SIMD issues an instruction per four
// cycles at best, so the instructions of a step are the time (64 blocks of two
// 128 x 128 planes: a wavefront issues in 46 % of its cycles): the factor
// operands lie in anti-diagonal order (lane l's entry of a step is contiguous),
// addresses advance by constants, every access goes through a buffer
// descriptor whose bounds check drops the lanes off the block (no selects of
// addresses, no sink stores, no branches), all ring slots are immediate
// offsets, and both streams are loaded two groups ahead.  With one block per
// CU (256 planes of 256 x 256) HBM bounds it: 1.3 GB of traffic at 4.70 TB/s,
// near a copy's 4.75.  With six wavefronts a block on four SIMDs (80 blocks of
// two 160 x 160 planes) a wavefront issues in 22 % of its cycles and waits to
// issue in 55 %, at 2.1 TB/s: neither HBM nor the instruction count, but SIMDs
// that two wavefronts share and a barrier of all six every eight steps.
// Measured, one apply, against the kernels before (a line form for whole lines
// and planes with addresses selected per lane; level-scheduled sweeps for the
// others): 64 blocks of two 128 x 128 planes ILU(0) 157 -> 89 us; 256 planes of
// 256 x 256 with the fused update 388 -> 351 us in the solve; 80 blocks of two
// 160 x 160 planes D-ILU 813 -> 190 us; 256 blocks of 10 1/4 lines of 75 cells
// D-ILU 136 -> 22 us.  Double-double, 32 blocks of three 96 x 96 planes ILU(0)
// (level-scheduled before): 675 -> 268 us (350 with Dekker's products), bound
// by FP64 issue (a wavefront issues in 44 % of its cycles, and two of the four
// SIMDs hold two).
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "bj_sweep.hpp"
#include "dd.hpp"

namespace parcel {

namespace {

constexpr int kLG = 8;        // steps per group
constexpr int kLC = 24;       // steps kept per line (three groups)
// Elements per line in LDS.  An odd number of 8- or 16-byte elements puts the
// lines of a step in distinct banks.
constexpr int kLL = kLC + 1;
// Why 24: the chunk stored into the ring after group g (for use from group
// g + 1 on) overwrites the steps 24 before its own 8 g + 8 .. 8 g + 22, that
// is up to 8 g - 2, and group g + 1 reads steps 8 g - 1 and later.  The
// barrier stands before that store, so the group-g readers are done.

constexpr int kOOB = (int)0x80000000u;  // byte offset beyond every descriptor: loads give 0, stores are dropped

typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef __amdgpu_buffer_rsrc_t rsrc_t;

__device__ __forceinline__ rsrc_t make_rsrc(const void* p, long bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00027000);
}
__device__ __forceinline__ double buf_load(rsrc_t r, int off) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}
__device__ __forceinline__ double2 buf_load2(rsrc_t r, int off) {
  return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
__device__ __forceinline__ void buf_store(double v, rsrc_t r, int off) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, off, 0, 0);
}

// v of the lane below (DPP wave_shr:1); lane 0 receives `first`.
__device__ __forceinline__ double from_lane_below(double first, double v) {
  const long long o = __double_as_longlong(first), x = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp((int)o, (int)x, 0x138, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(x >> 32), 0x138, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
__device__ __forceinline__ dd from_lane_below(dd first, dd v) {
  return mkdd(from_lane_below(first.hi, v.hi), from_lane_below(first.lo, v.lo));
}

// Orders the LDS accesses of the lanes of one wavefront (no s_barrier: the
// lines are private to the wavefront between barriers).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// The arithmetic of a sweep: double, or dd as hi / lo arrays.
struct alignas(16) dd16 {
  double hi, lo;
};
template <int NV>
struct Num;
template <>
struct Num<1> {
  using V = double;
  using L = double;  // as it lies in LDS
  struct Vec {
    rsrc_t a;
    __device__ __forceinline__ V load(int off) const { return buf_load(a, off); }
    __device__ __forceinline__ void store(V v, int off) const { buf_store(v, a, off); }
  };
  struct Pair {
    V x, y;
  };
  struct Mat {
    rsrc_t a;
    __device__ __forceinline__ Pair load2(int off) const {
      const double2 v = buf_load2(a, off);
      return {v.x, v.y};
    }
    __device__ __forceinline__ V load1(int off) const { return buf_load(a, off); }
  };
  static __device__ __forceinline__ V get(const L& l) { return l; }
  static __device__ __forceinline__ L put(V v) { return v; }
  static __device__ __forceinline__ V sel(bool c, V a, V b) { return c ? a : b; }
  static __device__ __forceinline__ V num(double v) { return v; }
};
template <>
struct Num<2> {
  using V = dd;
  using L = dd16;
  struct Vec {
    rsrc_t a, b;
    __device__ __forceinline__ V load(int off) const { return mkdd(buf_load(a, off), buf_load(b, off)); }
    __device__ __forceinline__ void store(V v, int off) const {
      buf_store(v.hi, a, off);
      buf_store(v.lo, b, off);
    }
  };
  struct Pair {
    V x, y;
  };
  struct Mat {
    rsrc_t a, b;
    __device__ __forceinline__ Pair load2(int off) const {
      const double2 h = buf_load2(a, off), l = buf_load2(b, off);
      return {mkdd(h.x, l.x), mkdd(h.y, l.y)};
    }
    __device__ __forceinline__ V load1(int off) const { return mkdd(buf_load(a, off), buf_load(b, off)); }
  };
  static __device__ __forceinline__ V get(const L& l) { return mkdd(l.hi, l.lo); }
  static __device__ __forceinline__ L put(V v) { return {v.hi, v.lo}; }
  static __device__ __forceinline__ V sel(bool c, V a, V b) { return mkdd(c ? a.hi : b.hi, c ? a.lo : b.lo); }
  static __device__ __forceinline__ V num(double v) { return mkdd(v, 0.0); }
};

struct LineArgs {
  const LineBlock* blk;
  const LineWave* fw;
  const LineWave* bw;
  const double* c[2][2];  // [forward, backward][hi, lo]
  const double* e[2][2];
  int nx;
  long nxy;
  int wide;  // double-double: no fma products (a factor value is outside dd_fma_range)
};

// The couplings' stored order is fixed by the factor: the forward rows of
// both factors and the backward rows of D-ILU hold the plane neighbour
// first, then the line neighbour, then the cell neighbour (ILU(0) keeps the
// CRS order of the block, D-ILU walks its upper part downward); ILU(0)'s
// backward rows hold them the other way round.
// A wavefront's factor entries: one row of nl entries per step, lane l's entry
// of its cell c in row c + l modulo a period of at least nx and 8 rows.  A lane
// has at most one cell in each row of a period, and the lanes of a step share
// their row, so the rows hold nx nl entries and no gaps (a row for each of the
// nx + nl - 1 steps would be half empty at 64 lines of 64 cells, 8/9 at 8).  The
// step after the period's last goes back to row 0 between groups of kLG loads
// only: the first kLG - 1 rows stand a second time behind the period.  Few lines
// (all their steps fit that) keep a row per step.
inline int line_period(int nx) { return nx * ((kLG + nx - 1) / nx); }
inline bool line_wraps(int nx, int nl, int period) { return nx + nl - 1 > period + kLG - 1; }
inline int line_rows(int nx, int nl, int period) {
  return line_wraps(nx, nl, period) ? period + kLG - 1 : nx + nl - 1;
}

template <bool FWD, int MODE>
constexpr bool line_cell_first() { return !FWD && MODE == BJ_ILU0; }

// dd_div(z, 1) for the unit pivots of ILU(0)'s forward rows: with d = 1 the
// quotient's q1 is z.hi, its remainder 0 + z.lo and q2 that, so the result
// is z's parts added and split again (the same bits).  nan is 0, or NaN where
// dd_div's split of q1 overflows (|z.hi| beyond 2^996 or not finite).
__host__ __device__ __forceinline__ dd dd_div_one(dd z) {
  const double nan = 0.0 * (134217729.0 * z.hi);
  const double l = (0.0 + z.lo) + nan;
  const double h = z.hi + l;
  return mkdd(h, l - (h - z.hi));
}

// dd_mul and dd_div with the error of the hi parts' product from one fma in
// place of Dekker's split (2 operations for 17).  Both are that error exactly,
// so the bits are the same, while the split does not overflow and no partial
// product underflows: operands of [2^-480, 2^480] or 0 (a zero product gives
// +0 both ways).  The host tests the factor against that range, the sweep
// every value it produces (FmaRange), and a block with one outside is swept
// again from its input with dd_mul and dd_div.
__device__ __forceinline__ dd dd_mul_fma(dd a, dd b) {
  const double t1h = a.hi * b.hi;
  double t1l = fma(a.hi, b.hi, -t1h);
  t1l = t1l + (a.hi * b.lo + a.lo * b.hi);
  const double s1 = t1h + t1l;
  t1l = t1l - (s1 - t1h);
  return mkdd(s1, t1l);
}
__device__ __forceinline__ dd dd_div_fma(dd a, dd b) {
  const double q1 = a.hi / b.hi;
  double t1h = b.hi * q1;
  double t1l = fma(b.hi, q1, -t1h);
  t1l = t1l + (b.lo * q1);
  double s1 = t1h + t1l;
  t1l = t1l - (s1 - t1h);
  t1h = s1;
  s1 = a.hi - t1h;
  const double r1 = s1 - a.hi;
  double s2 = (a.hi - (s1 - r1)) - (t1h + r1);
  s2 = s2 - t1l;
  s2 = s2 + a.lo;
  const double q2 = (s1 + s2) / b.hi;
  const double h = q1 + q2;
  return mkdd(h, q2 - (h - q1));
}
constexpr int kFmaLo = (1023 - 480) << 20, kFmaHi = (1023 + 480) << 20;  // high words of 2^-480 and 2^480
inline bool dd_fma_range(double v) {
  unsigned long long u;
  __builtin_memcpy(&u, &v, 8);
  const int t = (int)((u >> 32) & 0x7fffffff);
  return (t >= kFmaLo && t < kFmaHi) || (u << 1) == 0;
}
// The smallest and largest magnitude seen, as high words less one: a zero
// wraps to the largest unsigned and the smallest signed number, and a
// subnormal whose high word is empty counts as 1.
struct FmaRange {
  unsigned lo = 0xffffffffu;
  int hi = -1;
  __device__ __forceinline__ void see(double v) {
    const unsigned l = (unsigned)__double2loint(v);
    const unsigned t = (((unsigned)__double2hiint(v) & 0x7fffffffu) | (l < 1u ? l : 1u)) - 1u;
    lo = t < lo ? t : lo;
    hi = (int)t > hi ? (int)t : hi;
  }
  __device__ __forceinline__ bool outside() const { return lo < (unsigned)(kFmaLo - 1) || hi >= kFmaHi - 1; }
};

// Of a sweep's groups, those that have steps (two at least: line_sweep peels
// them); the others bring the last chunks out of the ring.
__host__ __device__ __forceinline__ int line_sweep_groups(int ng) { return ng - 2 > 2 ? ng - 2 : 2; }

// One sweep of a block.  NR: steps the factor operands are loaded ahead.
// alphaf: the fused update's alpha, asked for once the first loads are out.
template <bool FWD, int MODE, bool FUSED, bool PL, bool MULTI, int NV, int NR, bool FMA = false, class AF>
__device__ __forceinline__ void line_sweep(const LineArgs& A, const LineBlock bk, const LineWave wv, int w, int W,
                                           const typename Num<NV>::Vec in, const typename Num<NV>::Vec out,
                                           const typename Num<NV>::Vec q, AF alphaf, typename Num<NV>::L* lds,
                                           FmaRange* rg = nullptr) {
  using N = Num<NV>;
  using V = typename N::V;
  constexpr bool kScale = !(FWD && MODE == BJ_ILU0);
  constexpr int NE = (PL ? 1 : 0) + (kScale ? 1 : 0);
  const int nx = A.nx;
  const int lane = threadIdx.x & 63;
  const int dir = FWD ? 0 : 1;
  const int ng = FWD ? bk.ngf : bk.ngb;
  constexpr int sg = FWD ? 1 : -1;
  // this lane's line: its cells inside the block are sweep cells xs .. xs + cnt - 1,
  // computed at steps tx .. tx + cnt - 1
  const int line = wv.row0 + sg * lane * nx;          // row of sweep cell 0
  const int ls = FWD ? line : line - (nx - 1);        // first row in natural order
  const int ra = max(ls, 0), rb = min(ls + nx, bk.len);
  const unsigned cnt = lane < wv.nl ? (unsigned)max(rb - ra, 0) : 0u;
  const int tl0 = wv.tw + lane;                       // step of cell 0
  const int tx = tl0 + (FWD ? ra - ls : ls + nx - rb);
  // double-double rows skip absent couplings: the first steps that have a
  // line and a plane neighbour (a cell neighbour exists after the first step)
  int tln = 0x3fffffff, tpn = 0x3fffffff;
  if constexpr (NV == 2) {
    if (lane > 0 || wv.hand >= 0) tln = tl0 + (FWD ? nx - ls : line + nx - bk.len + 1);
    if (PL && wv.plane >= 0) tpn = tl0 + (int)(FWD ? A.nxy - ls : line + A.nxy - bk.len + 1);
  }
  // the factor entries (line_period)
  const long ents = wv.back ? (long)(wv.back / 16 + (kLG - 1) * wv.nl) : wv.nl > 0 ? (long)(nx + wv.nl - 1) * wv.nl : 0;
  typename N::Mat mc, me;
  mc.a = make_rsrc(A.c[dir][0] + 2 * wv.ebase, ents * 16);
  me.a = make_rsrc(A.e[dir][0] + NE * wv.ebase, ents * 8 * NE);
  if constexpr (NV == 2) {
    mc.b = make_rsrc(A.c[dir][1] + 2 * wv.ebase, ents * 16);
    me.b = make_rsrc(A.e[dir][1] + NE * wv.ebase, ents * 8 * NE);
  }
  const int estep = wv.nl * 16;
  int eo = wv.first + lane * 16;  // of the next load
  // between groups of loads: a row from the period on goes back by it (one
  // before it would become a large unsigned number; lanes without a line may go
  // anywhere)
  auto wrap = [&]() { eo = (int)min((unsigned)eo, (unsigned)eo - (unsigned)wv.back); };
  // An absent coupling has coefficient +0 and neighbour value kZero, whose
  // product term is -0 in the row's fma (fma(-(+0), +0, z) forward and in
  // ILU(0)'s backward rows, fma(-0, +0, z) in D-ILU's), and z + (-0) == z for
  // every z, the signed zeros included: the same bits as skipping the term.
  // Cells off the block keep it, and the line of wavefronts without a
  // neighbour holds it.
  constexpr double kZero = (!FWD && MODE == BJ_DILU) ? -0.0 : 0.0;
  typename N::L* own = lds + (w * 64 + lane) * kLL;
  const typename N::L* zero = lds + 64 * W * kLL;
  const typename N::L* hnd = wv.hand >= 0 ? lds + (wv.hand * 64 + 63) * kLL : zero;
  const typename N::L* pln = wv.plane >= 0 ? lds + (wv.plane * 64 + lane) * kLL : zero;
  if (threadIdx.x < kLC) lds[64 * W * kLL + threadIdx.x] = N::put(N::num(kZero));
  if (MULTI) lds_barrier();
  else wave_lds_sync();
  // Staging: lane 8 j + c moves element c of the 8-row chunk of local line
  // 8 k + j, k = 0..7.  in(g) is the line's chunk (rows aligned to 8) that
  // holds the cell of step 8 g + 15: loaded during group g - 1, put into the
  // ring after group g and, swept by the end of group g + 2, stored during
  // group g + 3.  For k = 0 and
  // the g to load next: ri the byte offset of the element's row, ci 8 times
  // its cell; line 8 k is k (8 nx - 8) rows and -8 k cells away.
  const int sj = lane >> 3, sc = lane & 7;
  const int l0 = wv.row0 + sg * sj * nx;
  const int c15 = 15 - wv.tw - sj;
  const int rin0 = ((bk.lo + l0 + sg * c15) & ~7) - bk.lo + sc;
  const int cin0 = sg * (rin0 - l0);
  const unsigned kst = (unsigned)(sg * 64) * (unsigned)(nx - 1);  // (wraps only for lines that lenk masks)
  unsigned lenk[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) lenk[k] = 8 * k + sj < wv.nl ? 8u * (unsigned)nx : 0u;
  typename N::L* stg = lds + (w * 64 + sj) * kLL;
  // the element's ring slot in the chunks of group g and g + 1 (mod 3)
  int sa = cin0 + wv.tw + sj;  // group 0: 8 .. 22
  auto next_slot = [](int s) { return s + 8 >= kLC ? s + 8 - kLC : s + 8; };
  int sb = next_slot(sa);
  auto chunk_off = [&](int ri, int ci, int k) -> int {
    return (unsigned)(ci - 64 * k) < lenk[k] ? (int)((unsigned)ri + k * kst) : kOOB;
  };
  double alpha = 0.0;
  V va[2][8], vb[FUSED ? 2 : 1][FUSED ? 8 : 1];
  int mo[FUSED ? 2 : 1][FUSED ? 8 : 1];
  auto stage_load_k = [&](auto pc, int ri, int ci, int k) {
    constexpr int p = decltype(pc)::value;
    const int off = chunk_off(ri, ci, k);
    va[p][k] = in.load(off);
    if constexpr (FUSED) {
      vb[p][k] = q.load(off);
      mo[p][k] = off;
    }
  };
  auto stage_load = [&](auto pc, int ri, int ci) {
#pragma unroll
    for (int k = 0; k < 8; ++k) stage_load_k(pc, ri, ci, k);
  };
  auto stage_fill = [&](auto pc, int slot) {
    constexpr int p = decltype(pc)::value;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      V z0 = va[p][k];
      if constexpr (FUSED) {
        z0 = fma(-alpha, vb[p][k], z0);
        in.store(z0, mo[p][k]);
      }
      stg[8 * k * kLL + slot] = N::put(z0);
    }
  };
  struct Ops {
    typename N::Pair c;  // line and cell couplings in stored order
    V p, d;              // plane coupling, scale
  };
  Ops R[NR];
  int dt = -tx;  // t0 - tx of the current group
  auto load = [&](int du, Ops& o) {
    const int off = (unsigned)(dt + du) < cnt ? eo : kOOB;
    o.c = mc.load2(off);
    if constexpr (NE == 2) {
      const typename N::Pair v = me.load2(off);
      o.p = v.x;
      o.d = v.y;
    } else if constexpr (PL) {
      o.p = me.load1((int)((unsigned)off >> 1));
    } else if constexpr (kScale) {
      o.d = me.load1((int)((unsigned)off >> 1));
    }
    eo += estep;
  };
  V yprev = N::num(kZero);  // the thread's value of the previous step (its cell neighbour)
  auto step = [&](int u, V a, V hv, V pv, const Ops& o) -> V {
    const bool on = (unsigned)(dt + u) < cnt;
    const V yd = from_lane_below(hv, yprev);  // line neighbour
    V y;
    if constexpr (NV == 1) {
      if constexpr (!FWD && MODE == BJ_DILU) {
        // plane, line, cell; y = a - d * sum
        double z = PL ? fma(pv, o.p, 0.0) : fma(yd, o.c.x, 0.0);
        z = PL ? fma(yd, o.c.x, z) : z;
        z = fma(yprev, o.c.y, z);
        y = fma(-o.d, z, a);
      } else if constexpr (line_cell_first<FWD, MODE>()) {
        double z = fma(-yprev, o.c.x, a);
        z = fma(-yd, o.c.y, z);
        if (PL) z = fma(-pv, o.p, z);
        y = z / o.d;
      } else {
        double z = PL ? fma(-pv, o.p, a) : a;
        z = fma(-yd, o.c.x, z);
        z = fma(-yprev, o.c.y, z);
        y = MODE == BJ_ILU0 ? z : o.d * z;
      }
    } else {
      // the level-scheduled kernel's operations over the couplings a row has
      const bool hc = dt + u > 0, hl = dt + tx + u >= tln, hp = PL && dt + tx + u >= tpn;
      constexpr bool kAdd = !FWD && MODE == BJ_DILU;
      dd z = kAdd ? mkdd(0.0, 0.0) : a;
      auto term = [&](bool has, dd v, dd cf) {
        const dd prod = FMA ? dd_mul_fma(v, cf) : dd_mul(v, cf);
        z = N::sel(has, kAdd ? dd_add(z, prod) : dd_sub(z, prod), z);
      };
      if constexpr (line_cell_first<FWD, MODE>()) {
        term(hc, yprev, o.c.x);
        term(hl, yd, o.c.y);
        if (PL) term(hp, pv, o.p);
      } else {
        if (PL) term(hp, pv, o.p);
        term(hl, yd, o.c.x);
        term(hc, yprev, o.c.y);
      }
      if constexpr (MODE == BJ_ILU0) y = FWD ? dd_div_one(z) : FMA ? dd_div_fma(z, o.d) : dd_div(z, o.d);
      else y = FWD ? dd_mul(z, o.d) : dd_sub(a, dd_mul(o.d, z));
    }
    yprev = N::sel(on, y, N::num(kZero));
    if constexpr (FMA) rg->see(yprev.hi);
    return yprev;
  };
  int ri = rin0 * 8 - sg * 64, ci = cin0 * 8 - 64;  // of in(-1)
  int s0 = 0, s1 = 16, s2 = 8;                      // ring slots of groups g, g - 1, g - 2
  auto group = [&](auto pc) {
    constexpr int p = decltype(pc)::value;
    using Q = std::integral_constant<int, 1 - p>;
    wave_lds_sync();
    auto input = [&](int u, V& a, V& h, V& pl) {
      a = N::get(own[s0 + u]);
      if (MULTI) h = N::get(u > 0 ? hnd[s1 + u - 1] : hnd[s2 + 7]);
      if (PL) pl = N::get(u > 0 ? pln[s1 + u - 1] : pln[s2 + 7]);
    };
    // all of the group's inputs at its start; double-double (twice the
    // registers, and steps longer than an LDS round trip) one step ahead
    constexpr int NI = NV == 1 ? kLG : 2;
    V av[NI], hv[NI], pv[NI];
#pragma unroll
    for (int u = 0; u < NI; ++u) hv[u] = pv[u] = N::num(kZero);
#pragma unroll
    for (int u = 0; u < (NV == 1 ? kLG : 1); ++u) input(u, av[u], hv[u], pv[u]);
    // the swept chunk in(g - 3), four groups behind ri, out of the slots that
    // in(g) takes after the steps
    stage_load(Q{}, ri, ci);
    V ov[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) ov[k] = N::get(stg[8 * k * kLL + sa]);
    // a step, the factor operands NR steps ahead and an eighth of the swept
    // chunk (stores all after the steps: 160^3 on 80 blocks 199 -> 211 us, the
    // next chunk's loads spread over the steps too: 205 us)
#pragma unroll
    for (int u = 0; u < kLG; ++u) {
      if (NV == 2 && u + 1 < kLG) input(u + 1, av[(u + 1) % NI], hv[(u + 1) % NI], pv[(u + 1) % NI]);
      own[s0 + u] = N::put(step(u, av[u % NI], hv[u % NI], pv[u % NI], R[(p * kLG + u) % NR]));
      load(u + NR, R[(p * kLG + u) % NR]);
      out.store(ov[u], chunk_off(ri - sg * 4 * 64, ci - 4 * 64, u));
    }
    wrap();
    if (MULTI) lds_barrier();
    else wave_lds_sync();
    stage_fill(pc, sa);
    ri += sg * 64;
    ci += 64;
    dt += kLG;
    sa = sb;
    sb = next_slot(sb);
    const int s = s2;
    s2 = s1;
    s1 = s0;
    s0 = s;
  };
  // the chunks group 0 reads (in(-2) and in(-1)), then in(0) in flight
  using P0 = std::integral_constant<int, 0>;
  using P1 = std::integral_constant<int, 1>;
  stage_load(P0{}, ri - sg * 64, ci - 64);
  stage_load(P1{}, ri, ci);
  if constexpr (FUSED) alpha = alphaf();
  stage_fill(P0{}, sb);             // slot of group -2 == group 1
  stage_fill(P1{}, next_slot(sb));  // slot of group -1 == group 2
  ri += sg * 64;
  ci += 64;
  stage_load(P0{}, ri, ci);
  ri += sg * 64;
  ci += 64;
#pragma unroll
  for (int u = 0; u < NR; ++u) {
    load(u, R[u]);
    if (u + 1 == NR || (u + 1) % kLG == 0) wrap();
  }
  // the first two groups run outside the loop, so that the loop is entered
  // with the memory operations of two groups in flight on both of its paths
  // (the compiler's wait counts then match the steady state)
  group(P0{});
  group(P1{});
  const int nf = line_sweep_groups(ng);
  for (int g = 2; g < nf; g += 2) {
    group(P0{});
    if (g + 1 < nf) group(P1{});
  }
  // every step is done: the last chunks out of the ring (with whole groups here,
  // 65536 blocks of 2 x 8 cells took 570 us an apply, 433 now; 256 of ten lines of
  // 75 cells 23.4 and 21.7)
  for (int g = nf; g < ng; ++g) {
    wave_lds_sync();
#pragma unroll
    for (int k = 0; k < 8; ++k)
      out.store(N::get(stg[8 * k * kLL + sa]), chunk_off(ri - sg * 4 * 64, ci - 4 * 64, k));
    ri += sg * 64;
    ci += 64;
    sa = sb;
    sb = next_slot(sb);
  }
}

template <int NV>
__device__ __forceinline__ typename Num<NV>::Vec line_vec(const double* h, const double* l, const LineBlock& bk) {
  typename Num<NV>::Vec v;
  v.a = make_rsrc(h + bk.lo, (long)bk.len * 8);
  if constexpr (NV == 2) v.b = make_rsrc(l + bk.lo, (long)bk.len * 8);
  return v;
}

// One workgroup per block: forward then backward sweep.  The fused residual
// update computes alpha as k_bj_apply does, with gamma summed in the same
// order (partials j, j + kNT, ... per virtual thread j < kNT, wavefront sums,
// then the kWaves sums in order).  NTH: 64 (one wavefront per block: no
// barriers), 256 or 512 threads at most.
template <int MODE, int NTH, bool PL, bool FUSED>
__global__ void __launch_bounds__(NTH) k_bj_lines(LineArgs A, const double* rin, double* s, CGFuse fuse,
                                                  const int* skip) {
  extern __shared__ __align__(16) double lds_lines[];
  __shared__ double sh[kWaves];
  constexpr bool MULTI = NTH > 64;
  constexpr int NR = NTH > 256 ? 8 : 16;
  const int W = MULTI ? (int)(blockDim.x >> 6) : 1;
  const int w = MULTI ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  // the state and the tables are read together
  const int done = FUSED ? fuse.st->done_at : skip ? *skip : 0;
  const LineBlock bk = A.blk[blockIdx.x];
  const LineWave wf = A.fw[(long)blockIdx.x * W + w], wb = A.bw[(long)blockIdx.x * W + w];
  if (done != 0 && (!FUSED || done <= fuse.it)) return;
  auto alphaf = [&]() -> double {
    CGSlot* slot = &fuse.st->slot[fuse.it & 1];
    for (int vw = w; vw < kWaves; vw += W) {
      double a = 0.0;
      for (int j = vw * 64 + (threadIdx.x & 63); j < fuse.nb_prod; j += kNT) a = a + fuse.part_gamma[j];
      a = wave_sum(a);
      if ((threadIdx.x & 63) == 0) sh[vw] = a;
    }
    __syncthreads();
    double gamma = sh[0];
    for (int k = 1; k < kWaves; ++k) gamma = gamma + sh[k];
    const double alpha = slot->rho0 / gamma;
    if (blockIdx.x == 0 && threadIdx.x == 0) slot->alpha = alpha;
    return alpha;
  };
  auto none = []() -> double { return 0.0; };
  using Vec = Num<1>::Vec;
  const Vec vs = line_vec<1>(s, nullptr, bk);
  const Vec vr = line_vec<1>(FUSED ? fuse.r : rin, nullptr, bk);
  const Vec vq = line_vec<1>(FUSED ? fuse.q : rin, nullptr, bk);
  line_sweep<true, MODE, FUSED, PL, MULTI, 1, NR>(A, bk, wf, w, W, vr, vs, vq, alphaf, lds_lines);
  __syncthreads();  // forward values in memory before other threads' backward rows read them
  line_sweep<false, MODE, false, PL, MULTI, 1, NR>(A, bk, wb, w, W, vs, vs, vs, none, lds_lines);
}

template <int MODE, int NTH, bool PL>
__global__ void __launch_bounds__(NTH) k_bj_lines_dd(LineArgs A, const double* rh, const double* rl, double* sh,
                                                     double* sl, const int* skip) {
  extern __shared__ __align__(16) double lds_lines[];
  constexpr bool MULTI = NTH > 64;
  const int W = MULTI ? (int)(blockDim.x >> 6) : 1;
  const int w = MULTI ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  const int done = skip ? *skip : 0;
  const LineBlock bk = A.blk[blockIdx.x];
  const LineWave wf = A.fw[(long)blockIdx.x * W + w], wb = A.bw[(long)blockIdx.x * W + w];
  if (done) return;
  using Vec = Num<2>::Vec;
  const Vec vs = line_vec<2>(sh, sl, bk), vr = line_vec<2>(rh, rl, bk);
  dd16* lds = reinterpret_cast<dd16*>(lds_lines);
  // lds_lines asks for 16-byte alignment because of this: 8 bytes off, the
  // rings' 128-bit accesses took the apply from 284 (then) to 502 us
  __shared__ int outside;
  if (threadIdx.x == 0) outside = 0;
  auto none = []() -> double { return 0.0; };
  auto sweeps = [&](auto fma, FmaRange* rg) {
    line_sweep<true, MODE, false, PL, MULTI, 2, 4, decltype(fma)::value>(A, bk, wf, w, W, vr, vs, vs, none, lds, rg);
    __syncthreads();  // forward values in memory before other threads' backward rows read them
    line_sweep<false, MODE, false, PL, MULTI, 2, 4, decltype(fma)::value>(A, bk, wb, w, W, vs, vs, vs, none, lds, rg);
  };
  if (!A.wide) {
    FmaRange rg;
    sweeps(std::true_type(), &rg);
    if (__any(rg.outside())) outside = 1;
    __syncthreads();  // the flag, and the rings and stores before they are written again
    if (!outside) return;
  }
  sweeps(std::false_type(), nullptr);
}

size_t line_lds_bytes(int W, int parts) { return sizeof(double) * (size_t)parts * (64 * (size_t)W + 1) * kLL; }

constexpr size_t kLdsMax = 160 * 1024 - 256;  // dynamic LDS per workgroup on gfx950 (a few bytes are static)

// A block's pieces: for every plane the block touches, the first line of its
// slots and their number.
struct Pieces {
  int np = 0, wp = 0;  // pieces, wavefronts per piece
  bool coupled = false;
  std::vector<long> first;
  std::vector<int> ny;
};

// ny_plane lines per plane; a block longer than a plane couples its planes,
// whose slots then all start at the plane's first line (the same lane in
// every plane); the pieces of a shorter one start at their own first line.
Pieces pieces_of(int lo, int hi, long nx, long ny_plane, long nxy) {
  Pieces p;
  const long L0 = lo / nx, L1 = (hi - 1) / nx;
  const long z0 = L0 / ny_plane, z1 = L1 / ny_plane;
  p.np = (int)(z1 - z0 + 1);
  p.coupled = nxy > 0 && (long)hi - lo > nxy;
  int mx = 1;
  for (long z = z0; z <= z1; ++z) {
    long a = z * ny_plane, b = a + ny_plane;
    if (!p.coupled) {
      a = std::max(a, L0);
      b = std::min(b, L1 + 1);
    }
    p.first.push_back(a);
    p.ny.push_back((int)(b - a));
    mx = std::max(mx, (int)(b - a));
  }
  p.wp = (mx + 63) / 64;
  return p;
}

// Whether a dependency of the sweeps lies more than three levels back, beyond
// the LDS ring of the level-scheduled kernels.
bool beyond_ring(const std::vector<BlockSweep>& F, const std::vector<BlockSweep>& B) {
  int far = 0;
#pragma omp parallel for schedule(dynamic) reduction(| : far)
  for (size_t b = 0; b < F.size(); ++b)
    for (const BlockSweep* S : {&F[b], &B[b]}) {
      std::vector<int> lev(S->diag.size());
      for (size_t l = 0; l + 1 < S->lev_start.size(); ++l)
        for (int t = S->lev_start[l]; t < S->lev_start[l + 1]; ++t) lev[S->order[t]] = (int)l;
      for (size_t i = 0; i < lev.size() && !far; ++i)
        for (int q = S->ptr[i]; q < S->ptr[i + 1]; ++q)
          if (lev[i] - lev[S->dep[q]] > 3) far = 1;
    }
  return far != 0;
}

// Whether line wavefronts are the faster form: `waves` wavefronts a block and
// `groups` groups of steps in both sweeps, against the levels of both sweeps.
// Lines cost groups, however few lanes a group has at work, so many small
// planes in a block, or many wavefronts of two to eight cells a line, are the
// levels' (2048 blocks of eight 8 x 8 planes: 91 us level by level, 402 as
// lines; 1024 blocks of four 16 x 16 planes 70 and 103; 512 blocks of 512 lines
// of four cells 369 and 542), all else the lines' (up to 7 times faster).  The
// estimates, in us (less what both forms spend alike), take the longer of one
// block's chain, the work of all blocks on the device, and memory; fitted to 264
// FP64 and 105 double-double block shapes of 2^12 to 2^22 rows, within 16 % (rms).
// On these the form taken is the faster one, but for two double-double shapes
// where it costs 13 and 17 %.
bool line_pays(int device, const std::vector<BlockSweep>& F, const std::vector<BlockSweep>& B, int n, int waves,
               int groups, bool planes, int parts) {
  int cu = 0;
  if (hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cu < 1) return true;
  const double nblk = (double)F.size(), dd = parts == 2;
  int levels = 0, width = 1;
  for (size_t b = 0; b < F.size(); ++b) {
    int l = 0;
    for (const BlockSweep* S : {&F[b], &B[b]}) {
      l += std::max(0, (int)S->lev_start.size() - 1);
      for (size_t k = 0; k + 1 < S->lev_start.size(); ++k)
        width = std::max(width, S->lev_start[k + 1] - S->lev_start[k]);
    }
    levels = std::max(levels, l);
  }
  const double chain = groups * (planes ? 1.15 : 0.86) * (waves > 4 ? (dd ? 1.5 : 2.0) : 1.0);
  const double work = nblk * waves * groups / (4.0 * cu) * (planes ? 1.55 : 0.95);
  const double line = std::max({chain, work, n * 1.3e-5}) * (dd ? 3.0 : 1.0);
  auto level = [&](double slow) {
    return std::max({levels * (planes ? 0.37 : 0.29), nblk * levels / cu * (planes ? 0.24 : 0.19), n * 5.5e-5}) *
               (slow * (dd ? 2.5 : 1.0));
  };
  const double wide = width <= 256 ? 1.0 : width <= 512 ? 1.9 : 6.0;  // wavefronts a level needs; past 512 unpipelined
  return line <= level(wide) || (line <= level(2.0 * wide) && beyond_ring(F, B));
}

bool line_setup_at(Plan& P, const std::vector<BlockSweep>& F, const std::vector<BlockSweep>& B,
                   const std::vector<int>& blo, const std::vector<int>& bhi, int parts, bool forced, long nx,
                   long ny_plane, long nxy) {
  LineBJ& G = P.M.line;
  const int n = P.hA.n, nblk = (int)F.size(), X = (int)nx, period = line_period(X);
  const bool ilu0 = P.M.mode == BJ_ILU0;
  std::vector<Pieces> pc(nblk);
  int W = 1;
  bool pl = false;
  for (int b = 0; b < nblk; ++b) {
    if (bhi[b] <= blo[b] || (long)(bhi[b] - blo[b]) * 8 >= (1L << 31)) return false;
    pc[b] = pieces_of(blo[b], bhi[b], nx, ny_plane, nxy);
    const long waves = (long)pc[b].np * pc[b].wp;
    if (waves > 8) return false;
    W = std::max(W, (int)waves);
    pl = pl || pc[b].coupled;
  }
  if (line_lds_bytes(W, parts) > kLdsMax) return false;
  std::vector<LineBlock> blk(nblk);
  std::vector<LineWave> wv[2];
  for (auto& v : wv) v.assign((size_t)nblk * W, LineWave{0, 0, 0, -1, -1, 0, 0, 0});
  long ents = 0;
  for (int b = 0; b < nblk; ++b) {
    const Pieces& p = pc[b];
    int ng[2];
    for (int dir = 0; dir < 2; ++dir) {
      int nsteps = 1;
      long e = ents;
      for (int k = 0; k < p.np; ++k)
        for (int jw = 0; jw < p.wp; ++jw) {
          const int kn = dir == 0 ? k : p.np - 1 - k, w = k * p.wp + jw;
          LineWave& v = wv[dir][(size_t)b * W + w];
          v.nl = std::min(64, std::max(0, p.ny[kn] - 64 * jw));
          v.tw = 64 * jw + 8 * jw + (p.coupled ? 9 * k : 0);
          v.hand = jw > 0 ? w - 1 : -1;
          v.plane = p.coupled && k > 0 ? w - p.wp : -1;
          v.ebase = e;
          if (v.nl == 0) continue;
          // relative to lo: within (-2^31, 2^31) since a block spans less
          const long row0 = dir == 0 ? (p.first[kn] + 64L * jw) * nx : (p.first[kn] + p.ny[kn] - 64L * jw) * nx - 1;
          v.row0 = (int)(row0 - blo[b]);
          const long we = (long)line_rows(X, v.nl, period) * v.nl;
          if (we * 16 >= (1L << 30)) return false;
          // step tw in row 0 (of some repetition of the period)
          const bool wraps = line_wraps(X, v.nl, period);
          v.back = wraps ? period * v.nl * 16 : 0;
          v.first = (wraps ? (period - v.tw % period) % period : -v.tw) * v.nl * 16;
          e += we;
          nsteps = std::max(nsteps, v.tw + v.nl - 1 + X);
        }
      ng[dir] = std::max(2, (nsteps - 1) / kLG + 3);
      if (dir == 1) ents = e;  // both sweeps cut the lines alike: the same number of entries
    }
    blk[b] = LineBlock{blo[b], bhi[b] - blo[b], ng[0], ng[1]};
  }
  // Entries per row: 1.1 for whole lines of 64 cells, 1.9 at eight, 7.5 at two; a
  // block that couples planes also holds the lines of the planes it cuts.  Beyond
  // eight (64 bytes each in FP64, twice that in double-double) the tables would
  // dwarf the matrix and the level form is kept; small systems (up to 64 MB
  // more) are let through.
  if (ents > 8L * n + (1L << 20)) return false;
  if (!forced) {
    int groups = 0;
    for (const LineBlock& k : blk) groups = std::max(groups, line_sweep_groups(k.ngf) + line_sweep_groups(k.ngb));
    if (!line_pays(P.device, F, B, n, W, groups, pl, parts)) return false;
  }
  const int ne[2] = {(pl ? 1 : 0) + (ilu0 ? 0 : 1), (pl ? 1 : 0) + 1};
  const size_t pe = (size_t)std::max(parts, 1);
  std::vector<double> c[2][2], ev[2][2];
  for (int dir = 0; dir < 2; ++dir)
    for (size_t q = 0; q < pe; ++q) {
      c[dir][q].assign(2 * (size_t)ents, 0.0);
      ev[dir][q].assign((size_t)ne[dir] * (size_t)ents, 0.0);
    }
  const bool lo_on = P.M.dd_prec == 2;  // precision 1 applies the factors' hi parts only
  int bad = 0, wide = 0;
#pragma omp parallel for schedule(dynamic) reduction(| : bad, wide)
  for (int b = 0; b < nblk; ++b) {
    const Pieces& p = pc[b];
    const long z0 = (blo[b] / nx) / ny_plane;
    const int len = bhi[b] - blo[b];
    for (int i = 0; i < len && !bad; ++i) {
      const long g = (long)blo[b] + i, L = g / nx, z = L / ny_plane;
      const int x = (int)(g - L * nx), y = (int)(L - z * ny_plane), k = (int)(z - z0);
      const int j = (int)(L - p.first[k]);
      for (int dir = 0; dir < 2; ++dir) {
        const bool fwd = dir == 0;
        const BlockSweep& S = fwd ? F[b] : B[b];
        // the neighbours the sweep reads, in the kernel's order
        const long cn = fwd ? i - 1L : i + 1L, ln = fwd ? i - nx : i + nx, pn = fwd ? i - nxy : i + nxy;
        const bool hc = fwd ? x > 0 && cn >= 0 : x < X - 1 && cn < len;
        const bool hl = fwd ? y > 0 && ln >= 0 : y < ny_plane - 1 && ln < len;
        const bool hp = p.coupled && (fwd ? pn >= 0 : pn < len);
        const bool cell_first = !fwd && ilu0;
        long want[3];
        int nw = 0;
        if (cell_first) {
          if (hc) want[nw++] = cn;
          if (hl) want[nw++] = ln;
          if (hp) want[nw++] = pn;
        } else {
          if (hp) want[nw++] = pn;
          if (hl) want[nw++] = ln;
          if (hc) want[nw++] = cn;
        }
        if (S.ptr[i + 1] - S.ptr[i] != nw) { bad = 1; break; }
        const int jp = fwd ? j : p.ny[k] - 1 - j, ip = fwd ? x : X - 1 - x, kq = fwd ? k : p.np - 1 - k;
        const LineWave& v = wv[dir][(size_t)b * W + kq * p.wp + jp / 64];
        const int l = jp % 64;
        const bool wraps = line_wraps(X, v.nl, period);
        const int row = wraps ? (ip + l) % period : ip + l;
        const size_t e = (size_t)(v.ebase + (long)row * v.nl + l);
        const size_t again = wraps && row < kLG - 1 ? (size_t)period * v.nl : 0;  // its second place
        for (size_t q = 0; q < pe; ++q) {
          const std::vector<double>& sv = q ? S.val_lo : S.val;
          double vc = 0.0, vl = 0.0, vp = 0.0;
          for (int r = S.ptr[i], m = 0; r < S.ptr[i + 1]; ++r, ++m) {
            const long dp = S.dep[r];
            if (dp != want[m]) { bad = 1; break; }
            (hc && dp == cn ? vc : hl && dp == ln ? vl : vp) = q && !lo_on ? 0.0 : sv[r];
          }
          if (bad) break;
          auto put = [&](size_t at) {
            c[dir][q][2 * at] = cell_first ? vc : vl;
            c[dir][q][2 * at + 1] = cell_first ? vl : vc;
            double* t = ev[dir][q].data() + (size_t)ne[dir] * at;
            if (pl) *t++ = vp;
            if (ne[dir] > (pl ? 1 : 0)) *t = q ? (lo_on ? S.diag_lo[i] : 0.0) : S.diag[i];
          };
          put(e);
          if (again) put(e + again);
          if (pe == 2 && q == 0 && !(dd_fma_range(vc) && dd_fma_range(vl) && dd_fma_range(vp) && dd_fma_range(S.diag[i])))
            wide = 1;
        }
        if (bad) break;
      }
    }
  }
  if (bad) return false;
  G.blk.upload(blk, P.stream);
  G.fw.upload(wv[0], P.stream);
  G.bw.upload(wv[1], P.stream);
  for (int dir = 0; dir < 2; ++dir)
    for (size_t q = 0; q < pe; ++q) {
      G.c[dir][q].upload(c[dir][q], P.stream);
      G.e[dir][q].upload(ev[dir][q], P.stream);
    }
  PARCEL_HIP_CHECK(hipStreamSynchronize(P.stream));
  G.nx = X;
  G.nxy = pl ? nxy : 0;
  G.waves = W;
  G.entries = (pl ? 3 : 2) * ents;
  G.wide = wide != 0;
  G.on = true;
  return true;
}

LineArgs line_args(const LineBJ& G) {
  LineArgs A;
  A.blk = G.blk.p;
  A.fw = G.fw.p;
  A.bw = G.bw.p;
  for (int d = 0; d < 2; ++d)
    for (int q = 0; q < 2; ++q) {
      A.c[d][q] = G.c[d][q].p;
      A.e[d][q] = G.e[d][q].p;
    }
  A.nx = G.nx;
  A.nxy = G.nxy;
  A.wide = G.wide ? 1 : 0;
  return A;
}

// Launch with the dynamic LDS the workgroup needs (above 64 KiB a kernel has
// to be told first).
template <class K, class... Args>
void launch_lines(K kern, int nblocks, int waves, size_t shm, hipStream_t st, Args... args) {
  if (shm > 64 * 1024)
    PARCEL_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm));
  hipLaunchKernelGGL(kern, dim3(nblocks), dim3(64 * waves), shm, st, args...);
}

}  // namespace

// The block factors' pattern decides: the dependency offsets inside blocks
// are 1, nx and (blocks longer than a plane) nxy; where no block couples
// planes the matrix's first row gives the lines per plane, and if the rows do
// not fit that, every line but the first is tried with a line neighbour.
// PARCEL_HIP_BJ_LEVELS=1 in the environment keeps the level-scheduled apply, =0
// takes the lines also where line_pays would not.
bool line_setup(Plan& P, const std::vector<BlockSweep>& F, const std::vector<BlockSweep>& B,
                const std::vector<int>& blo, const std::vector<int>& bhi, int parts) {
  P.M.line = LineBJ();
  bool forced = false;
  if (const char* e = std::getenv("PARCEL_HIP_BJ_LEVELS")) {
    if (e[0] && e[0] != '0') return false;
    forced = e[0] == '0';
  }
  const int n = P.hA.n, nblk = (int)F.size();
  for (int b = 0; b + 1 < nblk; ++b)
    if (bhi[b] != blo[b + 1]) return false;
  long o1 = 0, o2 = 0;
  for (int b = 0; b < nblk; ++b)
    for (size_t i = 0; i + 1 < F[b].ptr.size(); ++i)
      for (int q = F[b].ptr[i]; q < F[b].ptr[i + 1]; ++q) {
        const long off = (long)i - F[b].dep[q];
        if (off <= 1 || off == o1 || off == o2) continue;
        if (!o1) o1 = off;
        else if (!o2) o2 = off;
        else return false;
      }
  if (o1 && o2 && o2 < o1) std::swap(o1, o2);
  if (o1 < 2 || o1 >= (1L << 24) || (o2 && o2 % o1)) return false;
  if (o2) return line_setup_at(P, F, B, blo, bhi, parts, forced, o1, o2 / o1, o2);
  // blocks without plane couplings: the other offset of the matrix's first
  // row, which has every forward neighbour of a grid
  const HostCSR& A = P.hA;
  long m2 = 0;
  for (int e = A.rowptr[0]; e < A.rowptr[1]; ++e) m2 = std::max(m2, (long)A.col[e]);
  const long all = (n + o1 - 1) / o1;
  if (m2 > o1 && m2 % o1 == 0 && line_setup_at(P, F, B, blo, bhi, parts, forced, o1, m2 / o1, 0)) return true;
  return line_setup_at(P, F, B, blo, bhi, parts, forced, o1, all, 0);
}

void line_apply(Plan& P, const double* r, double* s, const CGFuse* fuse, const int* skip) {
  const Precon& M = P.M;
  const LineBJ& G = M.line;
  const LineArgs A = line_args(G);
  CGFuse f;
  if (fuse) f = *fuse;
  const size_t shm = line_lds_bytes(G.waves, 1);
#define PARCEL_LINE_F(MODE, NTH, PL)                                                                              \
  do {                                                                                                            \
    if (fuse) launch_lines(k_bj_lines<MODE, NTH, PL, true>, M.nblocks, G.waves, shm, P.stream, A, r, s, f, skip); \
    else launch_lines(k_bj_lines<MODE, NTH, PL, false>, M.nblocks, G.waves, shm, P.stream, A, r, s, f, skip);     \
  } while (0)
#define PARCEL_LINE_P(MODE, NTH)              \
  do {                                        \
    if (G.nxy) PARCEL_LINE_F(MODE, NTH, true); \
    else PARCEL_LINE_F(MODE, NTH, false);     \
  } while (0)
#define PARCEL_LINE_W(MODE)                            \
  do {                                                 \
    if (G.waves == 1) PARCEL_LINE_F(MODE, 64, false);  \
    else if (G.waves <= 4) PARCEL_LINE_P(MODE, 256);   \
    else PARCEL_LINE_P(MODE, 512);                     \
  } while (0)
  if (M.mode == BJ_ILU0) PARCEL_LINE_W(BJ_ILU0);
  else PARCEL_LINE_W(BJ_DILU);
#undef PARCEL_LINE_W
#undef PARCEL_LINE_P
#undef PARCEL_LINE_F
}

void line_apply_dd(Plan& P, const double* rh, const double* rl, double* sh, double* sl, const int* skip) {
  const Precon& M = P.M;
  const LineBJ& G = M.line;
  LineArgs A = line_args(G);
  if (rh == sh || rl == sl) A.wide = 1;  // no input to sweep again from
  const size_t shm = line_lds_bytes(G.waves, 2);
#define PARCEL_LINE_K(MODE, NTH, PL) \
  launch_lines(k_bj_lines_dd<MODE, NTH, PL>, M.nblocks, G.waves, shm, P.stream, A, rh, rl, sh, sl, skip)
#define PARCEL_LINE_P(MODE, NTH)               \
  do {                                         \
    if (G.nxy) PARCEL_LINE_K(MODE, NTH, true); \
    else PARCEL_LINE_K(MODE, NTH, false);      \
  } while (0)
#define PARCEL_LINE_W(MODE)                           \
  do {                                                \
    if (G.waves == 1) PARCEL_LINE_K(MODE, 64, false); \
    else if (G.waves <= 4) PARCEL_LINE_P(MODE, 256);  \
    else PARCEL_LINE_P(MODE, 512);                    \
  } while (0)
  if (M.mode == BJ_ILU0) PARCEL_LINE_W(BJ_ILU0);
  else PARCEL_LINE_W(BJ_DILU);
#undef PARCEL_LINE_W
#undef PARCEL_LINE_P
#undef PARCEL_LINE_K
}

}  // namespace parcel
