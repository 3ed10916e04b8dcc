// cg_kernels.hpp -- the CG kernels, shared by the single-system solver
// (krylov.hip) and the batched solver (batched.hip).
//
// Every kernel takes a Bat: the per-system strides of vectors (vs) and of
// matrix values (as).  A batched launch has gridDim.y systems; system
// y = blockIdx.y works on vectors at y*vs, matrix values at y*as, partial
// sums at y*PART_N*kNBMax, its own CGState and history.  A single-system
// launch passes {0, 0} and gridDim.y = 1, so every offset is zero.  The
// arithmetic of a system never depends on the others.
#pragma once

#include "kernels.hpp"

namespace parcel {

struct Bat {
  long vs;  // vector stride between systems (0: one system)
  long as;  // matrix-value stride between systems
};

namespace {

__device__ __forceinline__ long sys_id() { return (long)blockIdx.y; }

// Owner index of this workgroup in the tiled layout.  Workgroups are dealt to
// the 8 XCDs round-robin by linear id, so with nb a multiple of 8 the owners
// of XCD k are made the contiguous range [k nb/8, (k+1) nb/8): a stencil's
// neighbour tiles then sit in the same XCD's L2.  A bijection on [0, nb):
// owner o still holds tiles o, o+nb, ... and writes partial slot o, so every
// sum is unchanged.
__device__ __forceinline__ int tile_owner() {
  const int nb = gridDim.x, b = blockIdx.x;
  return (nb & 7) ? b : (b & 7) * (nb >> 3) + (b >> 3);
}

template <class T>
__device__ __forceinline__ SellArgsT<T> sys_matrix(SellArgsT<T> A, const Bat& B) {
  A.val += sys_id() * B.as;
  return A;
}

// Matrix access of the fused CG kernel: the SELL-64 matrix, or a five-point
// stencil in natural order with symmetric couplings stored once per row.
template <class T, class G>
__device__ __forceinline__ T mat_row(const SellArgsT<T>& A, long i, G g) {
  return sell_row(A, i, g);
}

// Five-point stencil: c = a(i,i), e = a(i,i+1) = a(i+1,i), nn = a(i,i+nx) =
// a(i+nx,i); one system's arrays are vs apart.  A row sums its entries in
// the CSR order s, w, c, e, n (sell_row's order for that pattern), so the
// product is bitwise the SELL product when the matrix is exactly symmetric.
// DIA: nnd diagonals of n values each, diagonal j of row i at val[j*n + i],
// coupling row i to column i + off[j] (MatVec_dia, src/matrix.f90:2309-2379:
// every diagonal in stored order; entries whose column falls outside
// [0, n) are skipped).  A zero entry adds fma(0, x, t) = t, so the row sum
// equals the CRS row's without the zeros (dia2crs drops them).
template <class T>
struct DiaArgsT {
  const T* val;
  const int* off;
  int nnd;
  long n;
};
template <class T, class G>
__device__ __forceinline__ T mat_row(const DiaArgsT<T>& A, long i, G g) {
  T t = 0;
  for (int j = 0; j < A.nnd; ++j) {
    const long c = i + A.off[j];
    if (c >= 0 && c < A.n) t = fma(A.val[(long)j * A.n + i], g(c), t);
  }
  return t;
}
template <class T>
__device__ __forceinline__ DiaArgsT<T> sys_matrix(DiaArgsT<T> A, const Bat& B) {
  A.val += sys_id() * B.as;
  return A;
}

template <class T>
struct St5 {
  const T* c;
  const T* e;
  const T* nn;
  int nx, ny;
  FastDiv dx;  // by nx (a system's rows < 2^31)
};

template <class T, class G>
__device__ __forceinline__ T mat_row(const St5<T>& A, long i, G g) {
  const unsigned ui = (unsigned)i, yy = A.dx.div(ui);
  const int x = (int)(ui - yy * (unsigned)A.nx), y = (int)yy;
  T t = 0;
  if (y > 0) t = fma(A.nn[i - A.nx], g(i - A.nx), t);
  if (x > 0) t = fma(A.e[i - 1], g(i - 1), t);
  t = fma(A.c[i], g(i), t);
  if (x < A.nx - 1) t = fma(A.e[i], g(i + 1), t);
  if (y < A.ny - 1) t = fma(A.nn[i], g(i + A.nx), t);
  return t;
}

template <class T>
__device__ __forceinline__ St5<T> sys_matrix(St5<T> A, const Bat& B) {
  const long o = sys_id() * B.vs;
  A.c += o;
  A.e += o;
  A.nn += o;
  return A;
}

// Seven-point (3D) or five-point (2D) stencil in natural order with
// symmetric couplings stored once per row, for one system: c = a(i,i),
// e = a(i,i+1) = a(i+1,i), nn = a(i,i+nx) = a(i+nx,i), t = a(i,i+nxy) =
// a(i+nxy,i) (nxy = n for a single plane; t is then never read).  A row
// sums its entries in CSR order b, s, w, c, e, n, t over the neighbours the
// grid has, which is sell_row's order when every such neighbour is stored:
// the product equals the SELL product bit for bit.
template <class T>
struct St7 {
  const T* c;
  const T* e;
  const T* nn;
  const T* t;
  int nx, ny;
  long nxy, n;
  FastDiv dx, dy;  // by nx and ny (rows < 2^31)
};

template <class T, class G>
__device__ __forceinline__ T mat_row(const St7<T>& A, long i, G g) {
  const unsigned ui = (unsigned)i, l = A.dx.div(ui), q = A.dy.div(l);
  const int x = (int)(ui - l * (unsigned)A.nx), y = (int)(l - q * (unsigned)A.ny);
  T t = 0;
  if (i >= A.nxy) t = fma(A.t[i - A.nxy], g(i - A.nxy), t);
  if (y > 0) t = fma(A.nn[i - A.nx], g(i - A.nx), t);
  if (x > 0) t = fma(A.e[i - 1], g(i - 1), t);
  t = fma(A.c[i], g(i), t);
  if (x < A.nx - 1) t = fma(A.e[i], g(i + 1), t);
  if (y < A.ny - 1) t = fma(A.nn[i], g(i + A.nx), t);
  if (i + A.nxy < A.n) t = fma(A.t[i], g(i + A.nxy), t);
  return t;
}

template <class MT>
struct IsSt7 : std::false_type {};
template <class T>
struct IsSt7<St7<T>> : std::true_type {};

// Row i (< A.n) of the stencil form times g = beta p_old + s, mat_row's
// sum, with every operand loaded before the first product: an absent
// neighbour reads row i instead (an address inside the arrays) and a select
// drops its term, so a row is one round of independent loads.  The loads do
// not need beta: they are issued before it is known.
template <class T>
struct St7Row {
  T a[7], p[7], z[7];  // b, s, w, c, e, n, t
  bool has[7];
};
template <class T, class TZ>
__device__ __forceinline__ void st7_load(const St7<T>& A, long i, const T* __restrict__ po,
                                         const TZ* __restrict__ s, St7Row<T>& R) {
  const unsigned ui = (unsigned)i, l = A.dx.div(ui), q = A.dy.div(l);
  const int x = (int)(ui - l * (unsigned)A.nx), y = (int)(l - q * (unsigned)A.ny);
  const bool has[7] = {i >= A.nxy, y > 0, x > 0, true, x < A.nx - 1, y < A.ny - 1, i + A.nxy < A.n};
  const long nb[7] = {i - A.nxy, i - A.nx, i - 1, i, i + 1, i + A.nx, i + A.nxy};
  long at[7];
#pragma unroll
  for (int k = 0; k < 7; ++k) {
    R.has[k] = has[k];
    at[k] = has[k] ? nb[k] : i;
  }
  R.a[0] = A.t[at[0]];
  R.a[1] = A.nn[at[1]];
  R.a[2] = A.e[at[2]];
  R.a[3] = A.c[i];
  R.a[4] = A.e[i];
  R.a[5] = A.nn[i];
  R.a[6] = A.t[i];
#pragma unroll
  for (int k = 0; k < 7; ++k) {
    R.p[k] = po[at[k]];
    R.z[k] = (T)s[at[k]];
  }
}
// the row's sum; pn: p_new of the row itself
template <class T>
__device__ __forceinline__ T st7_sum(const St7Row<T>& R, T beta, T pn) {
  T t = 0;
#pragma unroll
  for (int k = 0; k < 7; ++k) {
    const T g = k == 3 ? pn : fma(beta, R.p[k], R.z[k]);
    t = R.has[k] ? fma(R.a[k], g, t) : t;
  }
  return t;
}

template <class T>
__device__ __forceinline__ St7<T> sys_matrix(St7<T> A, const Bat& B) {
  (void)B;  // single-system plans only
  return A;
}

__device__ __forceinline__ double* sys_part(double* part) { return part + sys_id() * (PART_N * kNBMax); }

// r = b - A x and the partials of <b,b>, <r,r> (calc_res_CRS,
// src/krylov_h.f90:343; pcg.f90:456-470)
// (T: vector and matrix value type; sums of products accumulate in double)
template <class T>
__global__ void __launch_bounds__(kNT) k_residual(int n, SellArgsT<T> A, const T* __restrict__ x,
                                                  const T* __restrict__ b, T* __restrict__ r, double* part,
                                                  Bat B) {
  __shared__ double sh[kWaves];
  const long so = sys_id() * B.vs;
  A = sys_matrix(A, B);
  x += so; b += so; r += so;
  part = sys_part(part);
  const int nb = gridDim.x;
  const long ntiles = ((long)n + kNT - 1) / kNT;
  double a0 = 0.0, a1 = 0.0;
  for (long k = tile_owner(); k < ntiles; k += nb) {
    const long i = k * kNT + threadIdx.x;
    if (i < n) {
      const T t = sell_row(A, i, [&](int c) { return x[c]; });
      const T bi = b[i];
      const T ri = bi - t;
      r[i] = ri;
      a0 = fma((double)bi, (double)bi, a0);
      a1 = fma((double)ri, (double)ri, a1);
    }
  }
  double s0 = block_sum(a0, sh);
  double s1 = block_sum(a1, sh);
  if (threadIdx.x == 0) {
    part[PART_BB * kNBMax + tile_owner()] = s0;
    part[PART_RR0 * kNBMax + tile_owner()] = s1;
  }
}

// partials of <x,y> into part[slot] (slot offset already applied by the
// caller; systems are PART_N*kNBMax apart)
template <class T, class TX = T>
__global__ void __launch_bounds__(kNT) k_dot_part(int n, const TX* __restrict__ x, const T* __restrict__ y,
                                                  double* part, Bat B) {
  __shared__ double sh[kWaves];
  const long so = sys_id() * B.vs;
  x += so; y += so;
  part = sys_part(part);
  const int nb = gridDim.x;
  const long ntiles = ((long)n + kNT - 1) / kNT;
  double a0 = 0.0;
  for (long k = tile_owner(); k < ntiles; k += nb) {
    const long i = k * kNT + threadIdx.x;
    if (i < n) a0 = fma((double)x[i], (double)y[i], a0);
  }
  double s0 = block_sum(a0, sh);
  if (threadIdx.x == 0) part[tile_owner()] = s0;
}

__global__ void __launch_bounds__(kNT) k_reduce_one(const double* part, int nb, double* out) {
  __shared__ double sh[kWaves];
  double v = reduce_part(part, nb, sh);
  if (threadIdx.x == 0) *out = v;
}

// bnorm, rnorm, rho0 of the initial residual (pcg.f90:456-490); slot 0.
// One workgroup per system.
__global__ void __launch_bounds__(kNT) k_cg_init(const double* part, int nb, CGState* st) {
  __shared__ double sh[kWaves];
  part = sys_part(const_cast<double*>(part));
  st += sys_id();
  const double bb = reduce_part(part + PART_BB * kNBMax, nb, sh);
  const double rr = reduce_part(part + PART_RR0 * kNBMax, nb, sh);
  const double rho0 = reduce_part(part + PART_RHO0 * kNBMax, nb, sh);
  if (threadIdx.x == 0) {
    st->bnorm = sqrt(bb);
    st->done_at = 0;
    st->niter = 0;
    st->iret = 0;
    CGSlot& s = st->slot[0];
    s.rho0 = rho0;
    s.alpha = 0.0;
    s.beta = 0.0;
    s.rnorm = sqrt(rr);
    s.itr = 0;
  }
}

// K1 of iteration `it`.  LB logical owners per workgroup: the tiled layout
// has nb = LB * gridDim.x owners; workgroup w runs owners tile_owner(w)*LB
// + j, j < LB, round by round (tile o + r*nb of every owner o in round r),
// and writes each owner's partial, so every sum equals the LB = 1 launch's
// while the partial reduction at the start is paid once per workgroup and
// LB rows per thread are in flight.  TZ: the stored type of the
// preconditioned residual s (float when an FP32 apply produced it: widened
// at use, exactly).
// rounds per trip of the stencil-form loop
constexpr int kSt7U = 2;

template <class T, int LB = 1, class MT = SellArgsT<T>, class TZ = T>
__global__ void __launch_bounds__(kNT) k_cg_spmv(int n, int it, int itrmax, double rtol, MT A,
                                                 T* __restrict__ x, const T* __restrict__ p_old,
                                                 const TZ* __restrict__ s, T* __restrict__ p_new,
                                                 T* __restrict__ q, double* part, CGState* st,
                                                 double* hist, int hist_cap, Bat B) {
  __shared__ double sh[kWaves * LB], sh2[kWaves * 2];
  st += sys_id();
  const int done = st->done_at;
  if (!(IsSt7<MT>::value && LB == 1) && done != 0 && done < it) return;
  const long so = sys_id() * B.vs;
  A = sys_matrix(A, B);
  x += so; p_old += so; s += so; p_new += so; q += so;
  part = sys_part(part);
  hist += sys_id() * hist_cap;
  const CGSlot& prev = st->slot[(it - 1) & 1];
  const double bnorm = st->bnorm;
  double alpha_prev, beta, rho0, rnorm;
  bool exit_loop = false;
  const int nb = gridDim.x * LB;
  const int o0 = tile_owner() * LB;
  const long ntiles = ((long)n + kNT - 1) / kNT;
  // stencil form: the first trip's operands, in flight while the state is read
  // and the partials are reduced (they depend on neither): a small system's
  // launch waits for one memory round trip less (with k_cg_update_pj's, 400
  // iterations of point-Jacobi CG: 200^2 4.68 -> 4.34 ms, 1000^2 13.8 -> 12.6,
  // 2048 x 1024 21.3 -> 19.8; a launch on 256^3 in FP32 169 -> 158 us, in FP64
  // 353 before and 358 now)
  constexpr bool kPre = IsSt7<MT>::value && LB == 1;
  constexpr int U = kSt7U;
  const long stride = (long)nb * kNT;
  St7Row<T> row[kPre ? U : 1];
  T xo[kPre ? U : 1];
  long ri[kPre ? U : 1];
  auto load_trip = [&](long base) {
    if constexpr (kPre) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        ri[u] = (base + o0) * kNT + threadIdx.x + u * stride;
        const long ic = ri[u] < n ? ri[u] : (long)n - 1;
        st7_load(A, ic, p_old, s, row[u]);
        xo[u] = x[ic];
      }
    }
  };
  load_trip(0);
  if (kPre && done != 0 && done < it) return;
  if (it == 1) {
    alpha_prev = 0.0;
    beta = 0.0;
    rho0 = prev.rho0;
    rnorm = prev.rnorm;
  } else {
    // pcg.f90:640-700: rnorm = sqrt(<r,r>); exit tests; beta = rho1/rho0
    double rho1, rr;
    reduce_part2(part + PART_RHO1 * kNBMax, part + PART_RR * kNBMax, nb, sh2, rho1, rr);
    rnorm = sqrt(rr);
    const double ratio = rnorm / bnorm;
    alpha_prev = prev.alpha;
    exit_loop = ratio < rtol || ratio > 1.0e8 || it - 1 >= itrmax;
    beta = rho1 / prev.rho0;
    rho0 = rho1;
  }
  if (exit_loop) {
    // loop ended after iteration it-1: final x += alpha p (pcg.f90:733)
    for (long base = 0; base < ntiles; base += nb) {
#pragma unroll
      for (int j = 0; j < LB; ++j) {
        const long i = (base + o0 + j) * kNT + threadIdx.x;
        if (i < n) x[i] = fma((T)alpha_prev, p_old[i], x[i]);
      }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      st->done_at = it;
      st->niter = it - 1;                       // pcg.f90:850
      st->iret = (it - 1 >= itrmax) ? 1 : 0;    // pcg.f90:851-855
      st->slot[it & 1].rnorm = rnorm;
      st->slot[it & 1].itr = it - 1;
    }
    return;
  }
  double acc[LB];
#pragma unroll
  for (int j = 0; j < LB; ++j) acc[j] = 0.0;
  if constexpr (kPre) {
    // kSt7U rounds per trip, every load of the trip issued before its first
    // product; each row's values and the partial's order are the loop's below
    for (long base = 0;;) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (ri[u] < n) {
          const T po = row[u].p[3];
          const T pn = fma((T)beta, po, row[u].z[3]);
          const T t = st7_sum(row[u], (T)beta, pn);
          x[ri[u]] = fma((T)alpha_prev, po, xo[u]);
          p_new[ri[u]] = pn;
          q[ri[u]] = t;
          acc[0] = fma((double)pn, (double)t, acc[0]);
        }
      }
      base += (long)U * nb;
      if (base >= ntiles) break;
      load_trip(base);
    }
  } else {
    for (long base = 0; base < ntiles; base += nb) {
#pragma unroll
      for (int j = 0; j < LB; ++j) {
        const long i = (base + o0 + j) * kNT + threadIdx.x;
        if (i < n) {
          const T po = p_old[i];
          x[i] = fma((T)alpha_prev, po, x[i]);
          const T pn = fma((T)beta, po, (T)s[i]);
          p_new[i] = pn;
          const T t = mat_row(A, i, [&](long c) { return fma((T)beta, p_old[c], (T)s[c]); });
          q[i] = t;
          acc[j] = fma((double)pn, (double)t, acc[j]);
        }
      }
    }
  }
  block_sum_n<LB>(acc, sh);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int j = 0; j < LB; ++j) part[PART_GAMMA * kNBMax + o0 + j] = acc[j];
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (it - 1 < hist_cap) hist[it - 1] = rnorm / bnorm;  // pcg.f90:512-518
    CGSlot& cur = st->slot[it & 1];
    cur.rho0 = rho0;
    cur.beta = beta;
    cur.rnorm = rnorm;
    cur.itr = it;
  }
}

// K2 of iteration `it` (point Jacobi or none): alpha; r -= alpha q;
// s = Dinv r; (rho1, rr) partials.  dinv == nullptr: s = r.
template <class T>
__global__ void __launch_bounds__(kNT) k_cg_update_pj(int n, int it, T* __restrict__ r, const T* __restrict__ q,
                                                      const T* __restrict__ dinv, T* __restrict__ s, double* part,
                                                      CGState* st, int nb_prod, Bat B) {
  __shared__ double sh[kWaves], sh2[kWaves * 2];
  st += sys_id();
  const int done = st->done_at;
  const long so = sys_id() * B.vs;
  r += so; q += so; s += so;
  if (dinv) dinv += so;
  part = sys_part(part);
  CGSlot& cur = st->slot[it & 1];
  const int nb = gridDim.x;
  const long ntiles = ((long)n + kNT - 1) / kNT;
  // the first tile's operands, in flight while the state is read and the
  // partials are reduced (256^2: 3.9 -> 3.6 us)
  long i = (long)tile_owner() * kNT + threadIdx.x;
  T r0 = 0, q0 = 0, d0 = 1;
  auto load = [&]() {
    if (i < n) {
      r0 = r[i];
      q0 = q[i];
      if (dinv) d0 = dinv[i];
    }
  };
  load();
  if (done != 0 && done <= it) return;
  const double gamma = reduce_part(part + PART_GAMMA * kNBMax, nb_prod, sh);
  const double alpha = cur.rho0 / gamma;  // pcg.f90:590-600
  if (blockIdx.x == 0 && threadIdx.x == 0) cur.alpha = alpha;
  double a[2] = {0.0, 0.0};
  for (long k = tile_owner();;) {
    if (i < n) {
      const T ri = fma(-(T)alpha, q0, r0);
      r[i] = ri;
      const T si = dinv ? ri * d0 : ri;
      s[i] = si;
      a[0] = fma((double)si, (double)ri, a[0]);
      a[1] = fma((double)ri, (double)ri, a[1]);
    }
    k += nb;
    if (k >= ntiles) break;
    i = k * kNT + threadIdx.x;
    load();
  }
  block_sum_n<2>(a, sh2);
  if (threadIdx.x == 0) {
    part[PART_RHO1 * kNBMax + tile_owner()] = a[0];
    part[PART_RR * kNBMax + tile_owner()] = a[1];
  }
}

// rho1 = <s,r>, rr = <r,r> partials (CG_calc_dot2, pcg.f90:30); LB logical
// owners per workgroup as in k_cg_spmv
template <class T, int LB = 1, class TZ = T>
__global__ void __launch_bounds__(kNT) k_cg_dot2(int n, int it, const TZ* __restrict__ s, const T* __restrict__ r,
                                                 double* part, const CGState* st, Bat B) {
  __shared__ double sh[kWaves * 2 * LB];
  st += sys_id();
  {
    const int d = st->done_at;
    if (d != 0 && d <= it) return;
  }
  const long so = sys_id() * B.vs;
  s += so; r += so;
  part = sys_part(part);
  const int nb = gridDim.x * LB;
  const int o0 = tile_owner() * LB;
  const long ntiles = ((long)n + kNT - 1) / kNT;
  double acc[2 * LB];
#pragma unroll
  for (int j = 0; j < 2 * LB; ++j) acc[j] = 0.0;
  for (long base = 0; base < ntiles; base += nb) {
#pragma unroll
    for (int j = 0; j < LB; ++j) {
      const long i = (base + o0 + j) * kNT + threadIdx.x;
      if (i < n) {
        const T ri = r[i];
        acc[j] = fma((double)s[i], (double)ri, acc[j]);
        acc[LB + j] = fma((double)ri, (double)ri, acc[LB + j]);
      }
    }
  }
  block_sum_n<2 * LB>(acc, sh);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int j = 0; j < LB; ++j) {
      part[PART_RHO1 * kNBMax + o0 + j] = acc[j];
      part[PART_RR * kNBMax + o0 + j] = acc[LB + j];
    }
  }
}

// alpha = rho0 / <p,q> (reduced from the SpMV's partials); r -= alpha q
// (pcg.f90:590-620) for a preconditioner applied in a separate step; LB
// logical owners per workgroup as in k_cg_spmv
template <class T, int LB = 1>
__global__ void __launch_bounds__(kNT) k_cg_axpy_r(int n, int it, T* __restrict__ r, const T* __restrict__ q,
                                                   double* part, CGState* st, int nb_prod, Bat B) {
  __shared__ double sh[kWaves];
  st += sys_id();
  {
    const int d = st->done_at;
    if (d != 0 && d <= it) return;
  }
  const long so = sys_id() * B.vs;
  r += so; q += so;
  part = sys_part(part);
  CGSlot& cur = st->slot[it & 1];
  const double gamma = reduce_part(part + PART_GAMMA * kNBMax, nb_prod, sh);
  const double alpha = cur.rho0 / gamma;  // pcg.f90:590-600
  if (blockIdx.x == 0 && threadIdx.x == 0) cur.alpha = alpha;
  const int nb = gridDim.x * LB;
  const int o0 = tile_owner() * LB;
  const long ntiles = ((long)n + kNT - 1) / kNT;
  for (long base = 0; base < ntiles; base += nb) {
#pragma unroll
    for (int j = 0; j < LB; ++j) {
      const long i = (base + o0 + j) * kNT + threadIdx.x;
      if (i < n) r[i] = fma(-(T)alpha, q[i], r[i]);
    }
  }
}

template <class T>
__global__ void __launch_bounds__(kNT) k_spmv(int n, SellArgsT<T> A, const T* __restrict__ x, T* __restrict__ y,
                                              Bat B) {
  const long so = sys_id() * B.vs;
  A = sys_matrix(A, B);
  x += so; y += so;
  const int nb = gridDim.x;
  const long ntiles = ((long)n + kNT - 1) / kNT;
  for (long k = tile_owner(); k < ntiles; k += nb) {
    const long i = k * kNT + threadIdx.x;
    if (i < n) y[i] = sell_row(A, i, [&](int c) { return x[c]; });
  }
}

constexpr Bat kOne{0, 0};

}  // namespace
}  // namespace parcel
