// wf_device.h -- device helpers shared by the step kernels (wf_kernels.hip)
// and their adjoint (wf_adjoint.hip): launch shapes, block reductions,
// the cubic-spline gradient factor, yield laws, amplitudes.
#pragma once
#include <math.h>

#include "wf_internal.h"

namespace wf {

#define WF_KERNEL __global__ __launch_bounds__(kBlock)

static inline int nblk(long long n) { return (int)((n + kBlock - 1) / kBlock); }

// grid of the neighbour-build kernels: they run every step but exit at once
// unless a search is due, so they use a modest grid with grid-stride loops
static inline int nblk_small(long long n) {
  const int b = nblk(n);
  return b < 1024 ? b : 1024;
}

// XCD-aware tile index.  The dispatcher hands consecutive workgroups to the
// 8 XCDs in turn and each XCD has its own L2; remapping makes XCD x walk one
// contiguous run of tiles, so a particle and its (Morton-adjacent)
// neighbours are fetched into the same L2.  Bijective for any grid size.
constexpr int kXcd = 8;
__device__ inline int xcd_tile(int b, int nb) {
  const int q = nb / kXcd, r = nb % kXcd;
  const int x = b % kXcd, k = b / kXcd;
  return x * q + (x < r ? x : r) + k;
}

// block partial of reduction slot `slot` (slot-major: coalesced in finalize)
__device__ inline double &part(const Dev &d, int slot, int block) {
  return d.partials[(long long)slot * d.nblocks + block];
}

// ---------------------------------------------------------------------------
// reductions

__device__ inline double wave_sum(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}
__device__ inline double wave_max(double v) {
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
  return v;
}
__device__ inline double wave_min(double v) {
  for (int off = 32; off > 0; off >>= 1) v = fmin(v, __shfl_xor(v, off, 64));
  return v;
}

// block reduction in a fixed order; result valid in thread 0
template <int OP>
__device__ inline double block_reduce(double v, double *sh) {
  v = OP == 0 ? wave_sum(v) : (OP == 1 ? wave_max(v) : wave_min(v));
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) sh[w] = v;
  __syncthreads();
  double r = 0.0;
  if (threadIdx.x == 0) {
    r = sh[0];
    for (int k = 1; k < (int)(blockDim.x >> 6); ++k)
      r = OP == 0 ? r + sh[k] : (OP == 1 ? fmax(r, sh[k]) : fmin(r, sh[k]));
  }
  __syncthreads();
  return r;
}

// lanes > 1: lane `sub` > 0 of each particle hands its NV partial sums to
// lane 0 through LDS (red: (LANES - 1) * NV * kBlock values); lane 0 adds
// them in lane order.  Every thread of the block must call this.
template <int LANES, int NV, typename R>
__device__ inline void combine_lanes(R (&v)[NV], R *red) {
  if constexpr (LANES > 1) {
    const int lane = threadIdx.x % kBlock, sub = threadIdx.x / kBlock;
    if (sub > 0)
      for (int c = 0; c < NV; ++c) red[((sub - 1) * NV + c) * kBlock + lane] = v[c];
    __syncthreads();
    if (sub == 0)
      for (int q = 1; q < LANES; ++q)
        for (int c = 0; c < NV; ++c) v[c] += red[((q - 1) * NV + c) * kBlock + lane];
  }
}

// Values handed from block to block inside one launch: written through to
// the memory the 8 XCDs share (their L2 caches are not coherent with each
// other) and read past the caches.  The writing wavefront calls stores_done()
// before it (or, after a barrier, another thread of its block) raises the
// counter that announces them.  A __threadfence() in its place writes the
// whole L2 back, which costs tens of microseconds.
template <typename T>
__device__ inline void put_agent(T *p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ inline T get_agent(const T *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// ---------------------------------------------------------------------------
// kernel functions (Source/Functions.cpp:74-87) and the neighbour predicate

// cubic spline gradient factor GK with GK * x_ij = grad_i W_ij (3D),
// Source/Functions.cpp:74-87:  GK = C/(q h) * P(q), C = 1/(pi h^4), so for
// q < 1: GK = c5 (-3 + 9/4 q) and for 1 <= q < 2: GK = c5 (-3/4 (2-q)^2) / q
// with c5 = 1/(pi h^5).  Reciprocals use the hardware estimate refined by two
// Newton steps (a few ulp from the correctly rounded quotient).
__device__ inline double rcp_d(double x) {
  double y = __builtin_amdgcn_rcp(x);
  double e = fma(-x, y, 1.0);
  y = fma(y, e, y);
  e = fma(-x, y, 1.0);
  return fma(y, e, y);
}
__device__ inline double rsqrt_d(double x) {
  double y = __builtin_amdgcn_rsq(x);
  double e = fma(-x * y, y, 1.0);
  y = fma(0.5 * y, e, y);
  e = fma(-x * y, y, 1.0);
  return fma(0.5 * y, e, y);
}

// kernel constants of smoothing length h in dimension dim: the gradient
// factor's c5 = 1/(pi h^5) in 3D, 10/(7 pi h^4) in 2D (plane strain; the
// cubic spline's C/h with C from Source/Functions.cpp:81)
struct KernH {
  double h, ih, c5;  // pair smoothing length, 1/h, c5
  int dim;
};
__device__ inline KernH kern_h(double h, int dim = 3) {
  KernH k;
  k.h = h;
  k.ih = rcp_d(h);
  k.dim = dim;
  const double ih2 = k.ih * k.ih;
  k.c5 = dim == 2 ? ih2 * ih2 * (10.0 / (7.0 * M_PI)) : ih2 * ih2 * k.ih * (1.0 / M_PI);
  return k;
}
// h of the pair (h_i + h_j)/2; reuses particle i's constants when h_j == h_i
__device__ inline KernH pair_h(const KernH &ki, double hi, double hj) {
  if (hj == hi) return ki;
  return kern_h((hi + hj) / 2, ki.dim);
}
__device__ inline double grad_kernel_r2(double r2, const KernH &k) {
  if (r2 == 0.0) return -3.0 * k.c5;
  const double ri = rsqrt_d(r2);
  const double q = r2 * ri * k.ih;
  if (q < 1.0) return k.c5 * (-3.0 + 2.25 * q);
  if (q < 2.0) {
    const double t = 2.0 - q;
    return k.c5 * (-0.75 * t * t) * (k.h * ri);
  }
  return 0.0;
}

// the same kernel math for either pair precision R (double or float):
// float uses the 1-ulp hardware reciprocal / reciprocal square root
__device__ inline double rcp_t(double x) { return rcp_d(x); }
__device__ inline float rcp_t(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ inline double rsqrt_t(double x) { return rsqrt_d(x); }
__device__ inline float rsqrt_t(float x) { return __builtin_amdgcn_rsqf(x); }

template <typename R>
struct KH {
  R h, ih, c5;
  int dim;
};
template <typename R>
__device__ inline KH<R> kern_h_t(R h, int dim = 3) {
  KH<R> k;
  k.h = h;
  k.ih = rcp_t(h);
  k.dim = dim;
  const R ih2 = k.ih * k.ih;
  k.c5 = dim == 2 ? ih2 * ih2 * (R)(10.0 / (7.0 * M_PI)) : ih2 * ih2 * k.ih * (R)(1.0 / M_PI);
  return k;
}
template <typename R>
__device__ inline KH<R> pair_h_t(const KH<R> &ki, R hi, R hj) {
  if (hj == hi) return ki;
  return kern_h_t<R>((hi + hj) / (R)2, ki.dim);
}
// both branches evaluated and selected (no divergent branch in the pair
// loops, so loads of later neighbours can be scheduled early); each branch
// rounds exactly as a branchy version would.  r2 = 0 makes ri infinite and q
// NaN, which selects nothing until the last select.
template <typename R>
__device__ inline R gk_t(R r2, const KH<R> &k) {
  const R ri = rsqrt_t(r2);
  const R q = r2 * ri * k.ih;
  const R inner = k.c5 * ((R)-3 + (R)2.25 * q);
  const R t = (R)2 - q;
  const R outer = k.c5 * ((R)-0.75 * t * t) * (k.h * ri);
  R g = q < (R)1 ? inner : (q < (R)2 ? outer : (R)0);
  return r2 == (R)0 ? (R)-3 * k.c5 : g;
}


// the FP64 row walks' gradient factor: its constants, and reciprocals
struct GkD {
  double ih, gin_a, gin_b, gout;  // 1/h, 2.25 c5, -3 c5, -0.75 c5 h
};
__device__ inline GkD gk_consts64(double h, int dim) {
  const KH<double> k = kern_h_t<double>(h, dim);
  return GkD{k.ih, 2.25 * k.c5, -3.0 * k.c5, -0.75 * k.c5 * h};
}
// 1/x and 1/sqrt(x): the hardware estimate (relative error d < 2^-23) and one
// third-order step, 1/x = y / (1 - e) = y (1 + e + e^2 + ...) with
// e = 1 - x y, and the series of (1 - e)^(-1/2): errors d^3 and below, under
// the rounding
__device__ inline double rcp3(double x) {
  const double y = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, y, 1.0);
  return fma(y, fma(e, e, e), y);
}
__device__ inline double rsqrt3(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}

// ---------------------------------------------------------------------------
// neighbour rows read in groups of four entries, and a tile's staged set

struct LdsRows {
  using G = ushort4;
  const ushort4 *row;
  long long np;
  int own;  // the particle's position in the staged set
  __device__ G group(int g) const { return row[(long long)g * np]; }
  __device__ G self() const {
    const unsigned short o = (unsigned short)own;
    return make_ushort4(o, o, o, o);
  }
};
struct HbmRows {
  using G = int4;
  const int4 *row;
  long long np;
  int own;  // the particle's index
  __device__ G group(int g) const { return row[(long long)g * np]; }
  __device__ G self() const { return make_int4(own, own, own, own); }
};
template <class G>
__device__ inline int entry(const G &c, int u) {
  return u == 0 ? (int)c.x : (u == 1 ? (int)c.y : (u == 2 ? (int)c.z : (int)c.w));
}

// Lane `sub` of LANES takes the group pairs (2k, 2k + 1) with k = sub,
// sub + LANES, ...: a row of ng groups costs its lanes ng groups in all
// (the second group of the last pair is a self group when ng is odd).  An
// iteration processes one pair, the next pair's row words loaded at its top
// so they are in flight while this pair is processed.  The iteration is one
// branch-free block (a branch between the groups lets the compiler sink the
// prefetch down to its use): a second group past the row's end is replaced
// by `self`, a group of four self entries, whose pair terms are zeros.  The
// groups beyond a row's end that the prefetch touches (at most 2 LANES + 1)
// lie inside the allocation (nb_rows keeps kRowSpare spare entries) and are
// never used.
// a, b: the lane's first two groups (rows.group(2 sub) and the next), which
// the kernels load before they stage the tile.
template <int LANES, class Rows, class F>
__device__ inline void walk_groups(const Rows &rows, int cnt, int sub, const typename Rows::G &self,
                                   typename Rows::G a, typename Rows::G b, F &&group_fn) {
  static_assert(4 * (2 * LANES + 2) <= kRowSpare, "prefetch stays in the row allocation");
  const int ng = (cnt + 3) >> 2;
  for (int g = 2 * sub; g < ng; g += 2 * LANES) {
    const typename Rows::G a2 = rows.group(g + 2 * LANES);
    const typename Rows::G b2 = rows.group(g + 2 * LANES + 1);
    // compiler-only barrier: the prefetch stays issued here (it may not be
    // re-formed as a load next to its use); emits no instruction
    asm volatile("" ::: "memory");
    group_fn(a);
    // the second group's loads are not hoisted over the first group's
    // arithmetic (that would hold both groups' records in registers)
    __builtin_amdgcn_sched_barrier(0);
    group_fn(g + 1 < ng ? b : self);
    // the register moves of the hand-over stay at the end of the iteration
    // (moved earlier they would wait for the prefetch)
    __builtin_amdgcn_sched_barrier(0);
    a = a2;
    b = b2;
  }
}


// all NT threads call put(p, j) for the entries of tile t's staged set (each
// thread's indices are loaded first), then meet at a barrier
template <int NT, class F>
__device__ inline void stage_set(const int *stage, int t, int U, F &&put) {
  constexpr int R = (kStageMax + NT - 1) / NT;
  const int *st = stage + (long long)t * kStageMax;
  int j[R];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int p = (int)threadIdx.x + q * NT;
    j[q] = p < U ? st[p] : -1;
  }
#pragma unroll
  for (int q = 0; q < R; ++q)
    if (j[q] >= 0) put((int)threadIdx.x + q * NT, j[q]);
  __syncthreads();
}

// amplitude::getValAtTime (Source/Domain.h:75-87)
__device__ inline double amp_value(const DevAmp &a, double t) {
  int i = a.n - 1;
  bool end = false;
  while (!end) {
    i--;
    if (i == 0 || t > a.t[i]) end = true;
  }
  return a.v[i] + (a.v[i + 1] - a.v[i]) / (a.t[i + 1] - a.t[i]) * (t - a.t[i]);
}

// pow for the yield laws: 0 and exponent 1 give exactly what pow gives,
// without its ~300 instructions (a particle that never yielded, T = T_t)
__device__ inline double pow_law(double x, double y) {
  if (x == 0.0 && y > 0.0) return 0.0;
  if (y == 1.0) return x;
  return pow(x, y);
}

__device__ inline double jc_yield(const DevMat &M, double strain, double sr, double T) {
  const double T_h = (T - M.jc_Tt) / (M.jc_Tm - M.jc_Tt);
  double f = 1.0;
  if (sr > M.jc_eps0) f = 1.0 + M.jc_C * log(sr / M.jc_eps0);
  return (M.jc_A + M.jc_B * pow_law(strain, M.jc_n)) * f * (1.0 - pow_law(T_h, M.jc_m));
}

// JohnsonCookDamage::CalcFractureStrain (Source/Material.cpp:76-92): the
// strain at fracture at plastic strain rate sr, triaxiality sig_as and
// temperature T, with the material's T_t, T_m and eps_0; capped at 10
__device__ inline double jc_fracture_strain(const DevMat &M, double sr, double sig_as, double T) {
  const double T_h = (T - M.jc_Tt) / (M.jc_Tm - M.jc_Tt);
  double f_sr = 1.0;
  double f_triax = M.dam[0];
  if (sr > M.jc_eps0) f_sr = 1.0 + log(sr / M.jc_eps0) * M.dam[3];
  if (sig_as < 1.5) f_triax = M.dam[0] + M.dam[1] * exp(M.dam[2] * sig_as);
  double ef = f_triax * f_sr * (1.0 + M.dam[4] * T_h);
  if (ef > 10.0) ef = 10.0;
  return ef;
}

// the damage weight of a pair: 1 - D_pair with D_pair = (D_i + D_j) / 2,
// clamped to 1 (the Johnson-Cook criterion's pair value, Source/Damage.cpp:
// 141-150; Source/InteractionAlt.cpp:54-60); not positive: the pair is
// skipped
__device__ inline double dam_weight(double Di, double Dj) {
  const double Dp = (Di + Dj) / 2.0;
  double f = 1.0;
  if (Dp > 0.0) f = 1.0 - Dp;
  if (f > 1.0) f = 1.0;
  return f;
}

__device__ inline double hol_yield(const DevMat &M, double strain) {
  if (strain + M.hol_eps0 > M.hol_eps1) return M.hol_K * pow(strain + M.hol_eps0, M.hol_m);
  return M.hol_sy0;
}

__device__ inline void cross_d(const double a[3], const double b[3], double c[3]) {
  c[0] = a[1] * b[2] - a[2] * b[1];
  c[1] = a[2] * b[0] - a[0] * b[2];
  c[2] = a[0] * b[1] - a[1] * b[0];
}

}  // namespace wf
