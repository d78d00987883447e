// wf_kernels.hip -- HIP kernels of the explicit SPH step for gfx950.
//
// Pair passes are gathers: one lane per particle walks its own neighbour
// row and accumulates in registers, so sums need no atomics and are
// deterministic for a fixed neighbour list.  Every directed pair is
// evaluated from both ends; the pair terms of the reference are odd or even
// under the swap (i,j) -> (j,i), so each end recovers the reference's
// contribution exactly (Source/InteractionAlt.cpp:12-640).
//
// Global reductions (reaction, energies, plastic work) are two-stage:
// fixed-order block partials, then one single-block finalize kernel.
#include <float.h>
#include <math.h>

#include <type_traits>

#include "wf_device.h"

namespace wf {

// What a gather reads of particle j: the FP64 state, or its FP32 shadows.
// FP64:  x = (x, y, z, h), v = (vx, vy, vz, m), m/rho and rho separate.
// FP32:  x = (x, y, z, m/rho), v = (vx, vy, vz, m), rho = m / (m/rho); the
//        smoothing length is uniform within a material (checked at set-up),
//        so the pair h is the particle's own and needs no gathered load.
template <bool MX>
struct Src;
template <>
struct Src<false> {
  using R = double;
  using R4 = double4;
  __device__ static R4 x(const Dev &d, int b, int j) { return d.xh[b][j]; }
  __device__ static R4 v(const Dev &d, int j) { return d.vm[j]; }
  __device__ static R h_own(const Dev &d, int b, int i, const R4 &xi) { return xi.w; }
  __device__ static KH<R> kh(const KH<R> &ki, const R4 &xi, const R4 &xj) { return pair_h_t<R>(ki, xi.w, xj.w); }
  __device__ static R vol(const Dev &d, int b, int j, const R4 &xj) { return d.vol[b][j]; }
  __device__ static R rho(const Dev &d, int b, int j, const R4 &xj, const R4 &vj) { return d.rho[b][j]; }
  // t = sigma_j / rho_j^2 formed as the reference forms it per pair
  __device__ static void srec(const Dev &d, int j, R t[6], R &rho) {
    const StressRec r = d.srec[j];
    for (int k = 0; k < 6; ++k) t[k] = r.s[k] * r.irho2;
    rho = r.rho;
  }
};
template <>
struct Src<true> {
  using R = float;
  using R4 = float4;
  __device__ static R4 x(const Dev &d, int b, int j) { return d.xhf[b][j]; }
  __device__ static R4 v(const Dev &d, int j) { return d.vmf[j]; }
  __device__ static R h_own(const Dev &d, int b, int i, const R4 &xi) { return (float)d.xh[b][i].w; }
  __device__ static KH<R> kh(const KH<R> &ki, const R4 &xi, const R4 &xj) { return ki; }
  __device__ static R vol(const Dev &d, int b, int j, const R4 &xj) { return xj.w; }
  __device__ static R rho(const Dev &d, int b, int j, const R4 &xj, const R4 &vj) { return vj.w * rcp_t(xj.w); }
  __device__ static void srec(const Dev &d, int j, R t[6], R &rho) {
    const StressRecF r = d.srecf[j];
    for (int k = 0; k < 6; ++k) t[k] = r.t[k];
    rho = r.rho;
  }
};

// CheckRadius (Source/Neighbour.cpp:361-372), evaluated without contraction
// so it rounds exactly as the host predicate does.
__device__ inline bool in_radius(const double4 a, const double4 b, double cellfac) {
#pragma clang fp contract(off)
  const double h = (a.w + b.w) / 2;
  const double dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z;
  const double r = sqrt(dx * dx + dy * dy + dz * dz);
  return (r / h) <= cellfac;
}

// ListGenerate's cell coordinate (Source/Neighbour.cpp:185-225)
__device__ inline int cell_coord(double x, double blpf, double cs, int cn) {
  double f = floor((x - blpf) / cs);
  if (!(f >= 0.0)) return 0;  // also catches NaN
  if (f >= (double)cn) return cn - 1;
  return (int)f;
}

// velocity of each plane and of its particles at the step's time
// (UserAcc's BC loop and the contact-mesh branch, Source/WeldForm.cpp:67-119)
__device__ inline void rigid_bc(const Dev &d, const BcTable &bc, int r) {
  if (r >= d.nrig) return;
  const int m = d.rmesh[r];
  const int zone = d.mesh_zone[m];
  bool set = false, wset = false;
  double v[3] = {0, 0, 0}, w[3] = {0, 0, 0};
  for (int b = 0; b < bc.n; ++b) {
    if (bc.zone[b] != zone || bc.type[b] != 0) continue;
    if (bc.value_type[b] == 1) {
      if (bc.amp[b] < 0) continue;
      const double f = bc.amp_factor[b] * amp_value(d.amps[bc.amp[b]], d.flags->time);
      for (int k = 0; k < 3; ++k) v[k] = f * bc.v[b][k];
    } else {
      for (int k = 0; k < 3; ++k) v[k] = bc.v[b][k];
      // SetRotAxisVel: constant BCs only (Source/WeldForm.cpp:97-101)
      for (int k = 0; k < 3; ++k) w[k] = bc.w[b][k];
      wset = true;
    }
    set = true;
  }
  if (!set) return;
  d.rv[r] = make_double4(v[0], v[1], v[2], 0.0);
  if (r == d.mesh_elem0[m]) {
    d.mv[m] = make_double4(v[0], v[1], v[2], 0.0);
    if (wset) d.mw[m] = make_double4(w[0], w[1], w[2], 0.0);
  }
}

// ---------------------------------------------------------------------------
// neighbour schedule (Source/SolverLeapfrog.cpp:160-201, 347-356)

// rigid: the planes' velocities of the step too (any thread's share)
WF_KERNEL void k_schedule(Dev d, int force, int rigid, BcTable bc) {
  if (rigid) rigid_bc(d, bc, blockIdx.x * kBlock + threadIdx.x);
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  DevFlags *f = d.flags;
  const int isfirst = f->step == 0;
  const int mx = f->yielded;
  int search = 0, periodic = 0;
  if (force) {
    search = periodic = 1;
  } else {
    // with damage: no search when yielding starts, and ts_i = 1 after the
    // first step, so the first step's search is the last
    // (Source/SolverLeapfrog.cpp:160-171)
    if (d.damage && !isfirst) f->ts_i = 1;
    if (!d.damage && mx && !f->isyielding) {
      search = 1;
      f->isyielding = 1;
      f->cleared = 0;
    } else if ((mx || isfirst) && f->ts_i == 0 && f->cleared) {
      search = periodic = 1;
      f->cleared = 0;
    }
  }
  f->step_yield = mx;
  f->do_search = search;
  // CalcGradCorrMatrix follows the periodic search and runs on the first
  // step, not after the first-yield search (Source/SolverLeapfrog.cpp:160-212)
  f->gc_due = d.gc_on && (periodic || isfirst);
  if (search) {
    f->nb_searches += 1;
    f->max_count = 0;
    f->directed_pairs = 0;
  }
}

// ---------------------------------------------------------------------------
// neighbour build: counting sort of the particles (and of the rigid contact
// particles) by reference cell, then one lane per particle scans the 27
// surrounding cells with the exact predicate.  A search step runs
// k_cell_hist, k_scan, k_scatter, k_cell_sort, k_build_nbr and, with LDS
// staging, k_stage; on other steps each of them returns at once.

__device__ inline int cell_of(const Dev &d, const double4 x) {
  const int cx = cell_coord(x.x, d.blpf[0], d.cellsize[0], d.cellno[0]);
  const int cy = cell_coord(x.y, d.blpf[1], d.cellsize[1], d.cellno[1]);
  const int cz = cell_coord(x.z, d.blpf[2], d.cellsize[2], d.cellno[2]);
  return (cx * d.cellno[1] + cy) * d.cellno[2] + cz;
}
// the particle's cell in the SPH search grid
__device__ inline int scell_of(const Dev &d, const double4 x) {
  const int cx = cell_coord(x.x, d.blpf[0], d.scellsize[0], d.scellno[0]);
  const int cy = cell_coord(x.y, d.blpf[1], d.scellsize[1], d.scellno[1]);
  const int cz = cell_coord(x.z, d.blpf[2], d.scellsize[2], d.scellno[2]);
  return (cx * d.scellno[1] + cy) * d.scellno[2] + cz;
}

// The order of a pair's particles in the reference's list: "first" is the
// particle whose cell the pair was found from (Source/Neighbour.cpp:418-477),
// the higher index within one cell, else the particle whose half stencil
// holds the other, i.e. with the cells' offset (dx, dy, dz) = cell_j - cell_i,
// each -1, 0 or 1: dz = 1, or dz = 0 and dy = 1, or dz = dy = 0 and dx = 1.
// That is the sign of dx + 3 dy + 9 dz, so one comparison of these keys
// decides: i is first where key_j > key_i.
__device__ inline long long thermal_key(const Dev &d, int c, int perm) {
  const int nz = d.cellno[2], ny = d.cellno[1];
  const int cz = c % nz, cy = (c / nz) % ny, cx = c / (nz * ny);
  return ((long long)(cx + 3 * cy + 9 * cz) << 32) | (unsigned)(0x7fffffff - perm);
}

// threads 0..n-1: the SPH particles; n..n+nrig-1: the rigid particles.
// The counts are zero on entry (allocation, then cleared by k_cell_sort
// once a search has consumed them).
// z-slice (quarter of the cell height) of a record with FP32 offset z from
// its cell's lower face: the floor of z / (cell height / 4), clamped into
// the cell (a particle clamped into a boundary cell, or one that rounds
// onto a face, counts in the nearest slice)
__device__ inline int z_slice(float z, float inv_hz) {
  const float q = z * inv_hz;
  return q < 1.f ? 0 : (q < 2.f ? 1 : (q < 3.f ? 2 : 3));
}

// The counter's old value is the particle's place among its cell's
// particles (in atomic order; k_cell_sort fixes the order).  Also records
// each SPH particle's z-slice in its search cell (offset
// rounded to FP32 exactly as k_cell_sort's records are) and, per block, the
// largest SPH h (its FP32 bits; h > 0, so the bits order as the values)
// for the candidate pruning of k_build_nbr.
WF_KERNEL void k_cell_hist(Dev d, int cur) {
  if (!d.flags->do_search) return;
  __shared__ unsigned hw[kBlock / 64];
  const int i = blockIdx.x * kBlock + threadIdx.x;
  const int lane = threadIdx.x & 63;
  unsigned hb = 0;
  int c = -1;
  if (i < d.n) {
    const double4 x = d.xh[cur][i];
    hb = __float_as_uint((float)x.w);
    const int rc = cell_of(d, x);
    d.cell[i] = rc;
    if (d.thermal) d.tkey[i] = thermal_key(d, rc, d.perm[i]);
    c = scell_of(d, x);
    d.scell[i] = c;
    const int cz = c % d.scellno[2];
    const double oz = d.blpf[2] + cz * d.scellsize[2];
    d.sslice[i] = (unsigned char)z_slice((float)(x.z - oz), 4.f / (float)d.scellsize[2]);
  }
  // one atomic per run of consecutive lanes in the same cell (the particles
  // are in Morton order, so a wavefront's lanes share few cells): the run's
  // first lane adds the run length, each lane takes the old count plus its
  // place in the run
  {
    const int cprev = __shfl_up(c, 1, 64);
    const unsigned long long heads = __ballot(lane == 0 || cprev != c);
    const unsigned long long upto = lane == 63 ? ~0ull : ((1ull << (lane + 1)) - 1);
    const int start = 63 - __clzll(heads & upto);
    const unsigned long long above = heads & ~upto;
    const int end = above ? __ffsll((long long)above) - 1 : 64;
    int base = 0;
    if (c >= 0 && lane == start) base = atomicAdd(&d.cell_count[c], end - start);
    base = __shfl(base, start, 64);
    if (c >= 0) d.srank[i] = base + (lane - start);
  }
  if (i >= d.n && i - d.n < d.nrig) {
    const int r = i - d.n;
    const int c = cell_of(d, d.rx[r]);
    d.rcell[r] = c;
    d.rrank[r] = atomicAdd(&d.rcount[c], 1);
  }
  for (int off = 32; off > 0; off >>= 1) hb = max(hb, (unsigned)__shfl_xor((int)hb, off, 64));
  if ((threadIdx.x & 63) == 0) hw[threadIdx.x >> 6] = hb;
  __syncthreads();
  if (threadIdx.x == 0 && blockIdx.x < d.nblocks) {
    unsigned m = hw[0];
    for (int w = 1; w < kBlock / 64; ++w) m = max(m, hw[w]);
    d.hblk[blockIdx.x] = m;
  }
}

// inclusive scan of one value per lane across a wavefront
__device__ inline int wave_scan_incl(int v) {
  const int lane = threadIdx.x & 63;
  for (int off = 1; off < 64; off <<= 1) {
    int t = __shfl_up(v, off, 64);
    if (lane >= off) v += t;
  }
  return v;
}

// block-wide exclusive scan (blockDim.x <= 1024); returns the block total
// in *tot
__device__ inline int block_scan_excl(int v, int *sh, int *tot) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int inc = wave_scan_incl(v);
  if (lane == 63) sh[w] = inc;
  __syncthreads();
  if (w == 0) {
    int s = lane < (int)(blockDim.x >> 6) ? sh[lane] : 0;
    int si = wave_scan_incl(s);
    if (lane < (int)(blockDim.x >> 6)) sh[lane] = si - s;
    if (lane == (int)(blockDim.x >> 6) - 1) sh[32] = si;
  }
  __syncthreads();
  int r = inc - v + sh[w];
  *tot = sh[32];
  __syncthreads();
  return r;
}

// Cell starts of the counting sort in two levels: each block scans one
// chunk of kScanChunk cells (four per thread, one block scan) into in-chunk
// offsets (loc) and the chunk's total (tot); the block that finishes last (a
// ticket counter, reset by it) scans the chunk totals into chunk offsets
// (off) and the grand total (start[ncells]).  A cell starts at loc[c] +
// off[c / kScanChunk]; k_cell_sort writes that into start[c].
constexpr int kScanThreads = 256;
constexpr int kScanPer = 4;
static_assert(kScanChunk == kScanThreads * kScanPer, "a chunk is one block's four cells per thread");
__host__ __device__ inline int scan_chunks(long long ncells) { return (int)((ncells + kScanChunk - 1) / kScanChunk); }

__device__ inline void scan_chunk(const int *cnt, int *loc, int *tot, int ncells, int b, int *sh) {
  const int c0 = b * kScanChunk + threadIdx.x * kScanPer;
  int v[kScanPer], sum = 0;
#pragma unroll
  for (int k = 0; k < kScanPer; ++k) {
    v[k] = c0 + k < ncells ? cnt[c0 + k] : 0;
    sum += v[k];
  }
  int t;
  int off = block_scan_excl(sum, sh, &t);
#pragma unroll
  for (int k = 0; k < kScanPer; ++k) {
    if (c0 + k < ncells) loc[c0 + k] = off;
    off += v[k];
  }
  if (threadIdx.x == 0) put_agent(&tot[b], t);
}

// exclusive scan of the chunk totals written by the other blocks of the
// launch (read past the L1 cache) into off[0..nch), the sum into *end
__device__ inline void scan_totals(const int *tot, int *off, int nch, int *end, int *sh) {
  int carry = 0;
  for (int base = 0; base < nch; base += kScanThreads) {
    const int q = base + threadIdx.x;
    const int v = q < nch ? get_agent(&tot[q]) : 0;
    int t;
    const int e = block_scan_excl(v, sh, &t);
    if (q < nch) off[q] = carry + e;
    carry += t;
  }
  if (threadIdx.x == 0) *end = carry;
}

// blocks [0, ns): chunks of the search grid's counts; [ns, ns + nr): chunks
// of the rigid particles' counts (reference grid).  Each block also reduces
// a share of k_cell_hist's per-block largest h; the last block combines the
// shares into the search's largest h.
__global__ __launch_bounds__(kScanThreads) void k_scan(Dev d) {
  if (!d.flags->do_search) return;
  __shared__ int sh[34];
  __shared__ int last;
  const int ns = scan_chunks(d.sncells), nr = d.nrig ? scan_chunks(d.ncells) : 0, nb = ns + nr;
  const int b = blockIdx.x;
  if (b < ns) scan_chunk(d.cell_count, d.cell_loc, d.ctot, d.sncells, b, sh);
  else scan_chunk(d.rcount, d.rloc, d.rtot, d.ncells, b - ns, sh);
  const int per = (d.nblocks + nb - 1) / nb;
  unsigned hb = 0;
  for (int q = b * per + threadIdx.x; q < min(d.nblocks, (b + 1) * per); q += kScanThreads) hb = max(hb, d.hblk[q]);
  for (int o = 32; o > 0; o >>= 1) hb = max(hb, (unsigned)__shfl_xor((int)hb, o, 64));
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = (int)hb;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned m = 0;
    for (int w = 0; w < kScanThreads / 64; ++w) m = max(m, (unsigned)sh[w]);
    put_agent(&d.hred[b], m);
    stores_done();
    last = atomicAdd(&d.flags->scan_ticket, 1u) == (unsigned)(nb - 1);
  }
  __syncthreads();
  if (!last) return;
  scan_totals(d.ctot, d.coff, ns, d.cell_start + d.sncells, sh);
  if (nr) scan_totals(d.rtot, d.roff, nr, d.rstart + d.ncells, sh);
  hb = 0;
  for (int q = threadIdx.x; q < nb; q += kScanThreads)
    hb = max(hb, get_agent(&d.hred[q]));
  for (int o = 32; o > 0; o >>= 1) hb = max(hb, (unsigned)__shfl_xor((int)hb, o, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = (int)hb;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned m = 0;
    for (int w = 0; w < kScanThreads / 64; ++w) m = max(m, (unsigned)sh[w]);
    d.flags->hmax_bits = m;
    d.flags->scan_ticket = 0;
  }
}

// each particle to its place: its cell's start plus its in-cell rank
WF_KERNEL void k_scatter(Dev d) {
  if (!d.flags->do_search) return;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < d.n) {
    const int c = d.scell[i];
    d.sorted[d.cell_loc[c] + d.coff[c / kScanChunk] + d.srank[i]] = i;
  } else if (i - d.n < d.nrig) {
    const int r = i - d.n, c = d.rcell[r];
    d.rsorted[d.rloc[c] + d.roff[c / kScanChunk] + d.rrank[r]] = r;
  }
}

// where search cell c's records start (its in-chunk offset plus its chunk's)
// and end
__device__ inline int cell_first(const Dev &d, int c) { return d.cell_loc[c] + d.coff[c / kScanChunk]; }
__device__ inline int cell_end(const Dev &d, int c) {
  return c + 1 < d.sncells ? cell_first(d, c + 1) : d.cell_start[d.sncells];
}
// lower corner of search cell c
__device__ inline double3 cell_corner(const Dev &d, int c) {
  const int nz = d.scellno[2], ny = d.scellno[1];
  const int cz = c % nz, cy = (c / nz) % ny, cx = c / (nz * ny);
  return make_double3(d.blpf[0] + cx * d.scellsize[0], d.blpf[1] + cy * d.scellsize[1],
                      d.blpf[2] + cz * d.scellsize[2]);
}
// the candidate record of particle j at position p, offsets from corner o
__device__ inline void put_record(const Dev &d, int cur, int p, int j, const double3 &o) {
  const double4 x = d.xh[cur][j];
  d.sxyz[p] = make_float4((float)(x.x - o.x), (float)(x.y - o.y), (float)(x.z - o.z), (float)x.w);
  d.sinfo[p] = make_int2(j, d.group[j]);
}

// cell c (or none, c < 0) of 2-16 particles by the 16-lane segment of the
// wavefront that lane belongs to: each lane holds one particle and counts
// the segment's smaller keys; every lane of the wavefront calls this
__device__ inline void sort_small_cell(const Dev &d, int cur, int c, int lane) {
  const int seg = lane >> 4, sl = lane & 15;
  int s = 0, e = 0;
  if (c >= 0) {
    s = cell_first(d, c);
    e = cell_end(d, c);
  }
  const bool act = sl < e - s;
  int j = 0, zs = 0;
  if (act) {
    j = d.sorted[s + sl];
    zs = d.sslice[j];
  }
  const long long key = act ? ((long long)zs << 32) | (long long)j : 0x7fffffffffffffffLL;
  int rank = 0;
#pragma unroll
  for (int q = 0; q < 16; ++q) rank += __shfl(key, (seg << 4) + q, 64) < key ? 1 : 0;
  const int sh = seg << 4;
  const unsigned b0 = (unsigned)((__ballot(act && zs == 0) >> sh) & 0xffffu);
  const unsigned b1 = (unsigned)((__ballot(act && zs <= 1) >> sh) & 0xffffu);
  const unsigned b2 = (unsigned)((__ballot(act && zs <= 2) >> sh) & 0xffffu);
  if (act) {
    d.sorted[s + rank] = j;
    put_record(d, cur, s + rank, j, cell_corner(d, c));
  }
  if (c >= 0 && sl == 0) d.soff[c] = make_int4(s + __popc(b0), s + __popc(b1), s + __popc(b2), e);
}

// one cell of two or more particles, by the 64 lanes of a wavefront (lane =
// its lane)
__device__ inline void sort_cell(const Dev &d, int cur, int c, int lane) {
  const int s = cell_first(d, c), e = cell_end(d, c);
  const int cnt = e - s;
  const double3 o = cell_corner(d, c);
  if (cnt <= 64) {
    int j = 0, sl = 0;
    if (lane < cnt) {
      j = d.sorted[s + lane];
      sl = d.sslice[j];
    }
    const long long key = lane < cnt ? ((long long)sl << 32) | (long long)j : 0x7fffffffffffffffLL;
    int rank = 0;
    for (int l = 0; l < cnt; ++l) rank += __shfl(key, l, 64) < key ? 1 : 0;
    const unsigned long long b0 = __ballot(lane < cnt && sl == 0);
    const unsigned long long b1 = __ballot(lane < cnt && sl <= 1);
    const unsigned long long b2 = __ballot(lane < cnt && sl <= 2);
    if (lane < cnt) {
      d.sorted[s + rank] = j;
      put_record(d, cur, s + rank, j, o);
    }
    if (lane == 0)
      d.soff[c] = make_int4(s + __popcll(b0), s + __popcll(b1), s + __popcll(b2), e);
    return;
  }
  if (lane != 0) return;
  // key (slice, index) of each entry, held in sinfo while sorting
  for (int p = s; p < e; ++p) {
    const int j = d.sorted[p];
    d.sinfo[p] = make_int2(j, d.sslice[j]);
  }
  for (int a = s + 1; a < e; ++a) {
    const int2 v = d.sinfo[a];
    int b = a - 1;
    for (; b >= s; --b) {
      const int2 u = d.sinfo[b];
      if (u.y < v.y || (u.y == v.y && u.x < v.x)) break;
      d.sinfo[b + 1] = u;
    }
    d.sinfo[b + 1] = v;
  }
  int st[3] = {e, e, e};
  for (int p = e - 1; p >= s; --p) {
    const int2 k = d.sinfo[p];
    if (k.y >= 1) st[0] = p;
    if (k.y >= 2) st[1] = p;
    if (k.y >= 3) st[2] = p;
    d.sorted[p] = k.x;
    put_record(d, cur, p, k.x, o);
  }
  d.soff[c] = make_int4(st[0], st[1], st[2], e);
}

// per cell: write the cell's start, clear the counters for the next search,
// order the cell's particles by z-slice, then by index (cells hold ~10-30
// particles; the order, and with it every neighbour row, becomes
// independent of the atomic order), record where slices 1-3 start, and write
// the candidate records (FP32 offsets from the cell's lower corner, h,
// index, group) in cell order.  A wavefront takes cells in groups of
// kSortGroup: one lane per cell writes the start, clears the counter and
// finishes a cell of at most one particle; then the wavefront sorts the
// group's cells of 2-16 particles four at a time (sort_small_cell) and the
// larger ones one after another (sort_cell), so grids of mostly empty
// cells cost little.  The wavefronts, and the threads writing the
// rigid grid's starts, stride over the cells (a modest grid, so a step
// without a search exits early at little cost).  A wavefront works through its
// group's larger cells one after another, so the group is as small as the
// grid allows (16 cells per wavefront on a grid of 5 thousand took 45 us per
// search of 35k particles, one 9 us; 3.7k 40 and 7, 370k 55 and 27, 954k 71
// and 52).
constexpr int kSortGroup = 16, kSortBlocks = 8192;
WF_KERNEL void k_cell_sort(Dev d, int cur, int group) {
  if (!d.flags->do_search) return;
  if (d.nrig)
    for (int c = blockIdx.x * kBlock + threadIdx.x; c < d.ncells; c += gridDim.x * kBlock) {
      d.rstart[c] = d.rloc[c] + d.roff[c / kScanChunk];
      d.rcount[c] = 0;
    }
  const int lane = threadIdx.x & 63;
  const int nw = gridDim.x * (kBlock / 64);
  for (int base = (blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6)) * group; base < d.sncells;
       base += nw * group) {
    const int c = base + lane;
    const bool mine = lane < group && c < d.sncells;
    int cnt = 0;
    if (mine) {
      const int s = cell_first(d, c), e = cell_end(d, c);
      cnt = e - s;
      d.cell_start[c] = s;
      d.cell_count[c] = 0;
      if (cnt <= 1) {
        int4 so = make_int4(s, s, s, e);
        if (cnt == 1) {
          const int j = d.sorted[s], sl = d.sslice[j];
          put_record(d, cur, s, j, cell_corner(d, c));
          so = make_int4(s + (sl <= 0 ? 1 : 0), s + (sl <= 1 ? 1 : 0), s + (sl <= 2 ? 1 : 0), e);
        }
        d.soff[c] = so;
      }
    }
    // cells of 2-16 particles four at a time, one per 16-lane segment;
    // larger cells by the whole wavefront
    unsigned long long small = __ballot(mine && cnt >= 2 && cnt <= 16);
    unsigned long long big = __ballot(mine && cnt > 16);
    while (small) {
      int cq[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        cq[q] = small ? base + __ffsll((long long)small) - 1 : -1;
        small &= small - 1;
      }
      const int seg = lane >> 4;
      sort_small_cell(d, cur, seg == 0 ? cq[0] : (seg == 1 ? cq[1] : (seg == 2 ? cq[2] : cq[3])), lane);
    }
    while (big) {
      const int l = __ffsll((long long)big) - 1;
      big &= big - 1;
      sort_cell(d, cur, base + l, lane);
    }
  }
}

// One lane per particle (lanes in cell order) over the 27 cells around the
// particle's own, in cell order (each cell's particles by z-slice, then by
// index), so a row lists its neighbours in a fixed order (cells of the SPH
// search grid).  The 27 cells are 9 columns of up to three consecutive cell
// ids, whose candidates are one contiguous range of the cell-ordered
// records; of it only the slices within reach of the particle are walked
// (columns out of reach are skipped), four candidates at a time, their
// loads issued together.
// The radius test runs in FP32 on offsets from the cell corners (|error| <
// 1e-6 relative at the radius) and is trusted outside a band of 1e-4
// around it; inside the band, and for a particle lying far outside the grid
// (clamped into a boundary cell, where its FP32 offset loses digits), the
// exact FP64 predicate CheckRadius decides.
WF_KERNEL void k_build_nbr(Dev d, int cur) {
  if (!d.flags->do_search) return;
  __shared__ double sh[kBlock / 64];
  // lanes take the particles in cell order: a cell's particles walk the same
  // candidate ranges in step, so their loads are shared and their loops
  // agree
  const int ps = xcd_tile(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  const int i = ps < d.n ? d.sorted[ps] : ps;
  const long long np = d.npad;
  int4 *row = reinterpret_cast<int4 *>(d.nbr) + i;
  int4 pend = make_int4(i, i, i, i);  // the row's last four entries (the group being filled)
  int4 *wp = row;                     // where the group being filled goes
  int cnt = 0;
  if (i < d.n && d.group[i] >= 0) {
    const int g = d.group[i];
    const double4 xi = d.xh[cur][i];
    const int c = d.scell[i];
    const int nz = d.scellno[2], ny = d.scellno[1], nx = d.scellno[0];
    const int cz = c % nz, cy = (c / nz) % ny, cx = c / (nz * ny);
    const float csx = (float)d.scellsize[0], csy = (float)d.scellsize[1], csz = (float)d.scellsize[2];
    const float oxi = (float)(xi.x - (d.blpf[0] + cx * d.scellsize[0]));
    const float oyi = (float)(xi.y - (d.blpf[1] + cy * d.scellsize[1]));
    const float ozi = (float)(xi.z - (d.blpf[2] + cz * d.scellsize[2]));
    const float hi = (float)xi.w, hcf = 0.5f * (float)d.cellfac;
    const bool exact_all = fabsf(oxi) > 64.f * csx || fabsf(oyi) > 64.f * csy || fabsf(ozi) > 64.f * csz;
    const int az0 = cz > 0 ? cz - 1 : 0, az1 = cz + 1 < nz ? cz + 1 : nz - 1, m = az1 - az0;
    // every neighbour lies within ri of particle i: the pair radius
    // Cellfac (h_i + h_j) / 2 with h_j at most the largest h of the search,
    // widened by 1e-4 (FP32 rounding of these offsets is ~1e-7 of a cell)
    const float ri = hcf * (hi + __uint_as_float(d.flags->hmax_bits)) * 1.0001f, ri2 = ri * ri;
    const float inv_hz = 4.f / csz;  // the z-slices of k_cell_sort
    const int gmax = 4 * m + 3;      // last slice of the column
    // z of i from the lower faces of cells az0, az0 + 1, az0 + 2
    const float bz0 = (float)(cz - az0) * csz + ozi, bz1 = (float)(cz - az0 - 1) * csz + ozi,
                bz2 = (float)(cz - az0 - 2) * csz + ozi;
    for (int col = 0; col < 9; ++col) {
      const int dcx = col / 3 - 1, dcy = col % 3 - 1;
      const int ax = cx + dcx, ay = cy + dcy;
      if (ax < 0 || ax >= nx || ay < 0 || ay >= ny) continue;
      const float bx = (float)(cx - ax) * csx + oxi, by = (float)(cy - ay) * csy + oyi;
      const int cc0 = (ax * ny + ay) * nz + az0;
      // candidates of cells az0, az0 + 1, az0 + 2 start at s0, s1, s2
      const int s0 = d.cell_start[cc0], s1 = d.cell_start[cc0 + 1];
      const int s2 = m >= 1 ? d.cell_start[cc0 + 2] : s1;
      const int se = d.cell_start[cc0 + m + 1];
      // the column's records within reach: the column lies at least rho from
      // i across x and y (a face of i's own cell bounds it, clamped records
      // included), so only |z - z_i| <= sqrt(ri^2 - rho^2) can pair, which
      // is slices glo..ghi of the column (z from the bottom of cell az0)
      int lo = s0, hi_end = se;
      if (!exact_all) {
        const float gx = fmaxf(dcx < 0 ? oxi : (dcx > 0 ? csx - oxi : 0.f), 0.f);
        const float gy = fmaxf(dcy < 0 ? oyi : (dcy > 0 ? csy - oyi : 0.f), 0.f);
        const float rho2 = gx * gx + gy * gy;
        if (rho2 > ri2) continue;
        const float w = sqrtf(ri2 - rho2);
        const int glo = min(max((int)floorf((bz0 - w) * inv_hz), 0), gmax);
        const int ghi = min(max((int)floorf((bz0 + w) * inv_hz), 0), gmax);
        const int alo = glo >> 2, klo = glo & 3, ahi = ghi >> 2, khi = ghi & 3;
        const int4 ol = d.soff[cc0 + alo], oh = d.soff[cc0 + ahi];
        lo = klo == 0 ? (alo == 0 ? s0 : (alo == 1 ? s1 : s2)) : (klo == 1 ? ol.x : (klo == 2 ? ol.y : ol.z));
        hi_end = khi == 3 ? oh.w : (khi == 0 ? oh.x : (khi == 1 ? oh.y : oh.z));
      }
      // (the record arrays hold 4 spare entries, so a batch may read past
      // the range's end; those candidates are not valid)
      const int2 *fp = d.sinfo + lo;
      const float4 *qp = d.sxyz + lo;
      for (int pb = lo; pb < hi_end; pb += 4, fp += 4, qp += 4) {
        int2 f[4];
        float4 q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          f[u] = fp[u];
          q[u] = qp[u];
        }
        // compiler-only barrier: the four candidates' loads stay issued
        // together (not sunk into the accept branches); emits no instruction
        asm volatile("" ::: "memory");
        bool in[4], near[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int p = pb + u;
          const bool valid = (p < hi_end) & (f[u].x != i) & (f[u].y == g);
          const float bz = p >= s2 ? bz2 : (p >= s1 ? bz1 : bz0);
          const float dx = bx - q[u].x, dy = by - q[u].y, dz = bz - q[u].z;
          const float r2 = dx * dx + dy * dy + dz * dz;
          const float t = hcf * (hi + q[u].w);
          const float t2 = t * t;
          in[u] = valid & (r2 < t2);
          near[u] = valid & (exact_all | (fabsf(r2 - t2) <= 1e-4f * t2));
        }
        // the exact predicate decides the (rare) candidates in the band
        if (near[0] | near[1] | near[2] | near[3]) {
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (near[u]) in[u] = in_radius(xi, d.xh[cur][f[u].x], d.cellfac);
        }
        // append without branches: the group being filled shifts left and
        // the entry enters at w; a full group is stored (entries past max_nb
        // are only counted)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const bool take = in[u] && cnt < d.max_nb;
          pend.x = take ? pend.y : pend.x;
          pend.y = take ? pend.z : pend.y;
          pend.z = take ? pend.w : pend.z;
          pend.w = take ? f[u].x : pend.w;
          cnt += in[u] ? 1 : 0;
          if (take & ((cnt & 3) == 0)) {
            *wp = pend;
            wp += np;
          }
        }
      }
    }
  }
  if (i < d.n) {
    const int kept = cnt < d.max_nb ? cnt : d.max_nb;
    d.nnb[i] = kept;
    if (cnt > d.max_nb) d.flags->overflow = 1;
    // the pair passes read rows in groups of four: the rest of the last
    // group holds the particle itself (a pair term of exact zeros)
    // (the k = kept & 3 pending entries sit in the last k places of pend)
    if (kept & 3) {
      const int k = kept & 3;
      const int4 last = k == 1 ? make_int4(pend.w, i, i, i)
                               : (k == 2 ? make_int4(pend.z, pend.w, i, i) : make_int4(pend.y, pend.z, pend.w, i));
      *wp = last;
    }
  }
  // deterministic totals via block reduction + integer atomics
  const double bt = block_reduce<0>((double)cnt, sh);
  const double bm = block_reduce<1>((double)cnt, sh);
  if (threadIdx.x == 0) {
    atomicAdd((unsigned long long *)&d.flags->directed_pairs, (unsigned long long)bt);
    atomicMax(&d.flags->max_count, (int)bm);
  }
}

// The same rows with kBuildLanes lanes per particle, for models whose lanes of
// k_build_nbr would leave most of the chip idle: the first nine lanes form the
// nine columns' ranges together, then the lanes test as many candidates of a
// column at a time and append them in the records' order by a count of the
// lanes below.  Per search, one lane against 32 per particle: 58 and 16.5 us at
// 1.3k particles, 70 and 28 at 3.7k, but 66 and 214 at 35k.
constexpr int kBuildLanes = 32;
WF_KERNEL void k_build_nbr_wide(Dev d, int cur) {
  if (!d.flags->do_search) return;
  __shared__ double sh[kBlock / 64];
  const int sl = threadIdx.x & (kBuildLanes - 1), seg = threadIdx.x & 63 & ~(kBuildLanes - 1);
  const int ps = (int)((blockIdx.x * (long long)kBlock + threadIdx.x) / kBuildLanes);
  const int i = ps < d.n ? d.sorted[ps] : ps;
  const long long np = d.npad;
  const bool on = i < d.n && d.group[i] >= 0;
  const int ii = on ? i : 0;
  const int g = d.group[ii];
  const double4 xi = d.xh[cur][ii];
  const int c = d.scell[ii];
  const int nz = d.scellno[2], ny = d.scellno[1], nx = d.scellno[0];
  const int cz = c % nz, cy = (c / nz) % ny, cx = c / (nz * ny);
  const float csx = (float)d.scellsize[0], csy = (float)d.scellsize[1], csz = (float)d.scellsize[2];
  const float oxi = (float)(xi.x - (d.blpf[0] + cx * d.scellsize[0]));
  const float oyi = (float)(xi.y - (d.blpf[1] + cy * d.scellsize[1]));
  const float ozi = (float)(xi.z - (d.blpf[2] + cz * d.scellsize[2]));
  const float hi = (float)xi.w, hcf = 0.5f * (float)d.cellfac;
  const bool exact_all = fabsf(oxi) > 64.f * csx || fabsf(oyi) > 64.f * csy || fabsf(ozi) > 64.f * csz;
  const int az0 = cz > 0 ? cz - 1 : 0, az1 = cz + 1 < nz ? cz + 1 : nz - 1, m = az1 - az0;
  const float ri = hcf * (hi + __uint_as_float(d.flags->hmax_bits)) * 1.0001f, ri2 = ri * ri;
  const float inv_hz = 4.f / csz;
  const int gmax = 4 * m + 3;
  const float bz0 = (float)(cz - az0) * csz + ozi, bz1 = (float)(cz - az0 - 1) * csz + ozi,
              bz2 = (float)(cz - az0 - 2) * csz + ozi;
  // lane col < 9 of the particle: the column's records within reach (see
  // k_build_nbr), where its cells start and its offset from the particle
  int lo = 0, hi_end = 0, s1 = 0, s2 = 0;
  float bx = 0.f, by = 0.f;
  if (on && sl < 9) {
    const int dcx = sl / 3 - 1, dcy = sl % 3 - 1;
    const int ax = cx + dcx, ay = cy + dcy;
    if (ax >= 0 && ax < nx && ay >= 0 && ay < ny) {
      bx = (float)(cx - ax) * csx + oxi;
      by = (float)(cy - ay) * csy + oyi;
      const int cc0 = (ax * ny + ay) * nz + az0;
      const int s0 = d.cell_start[cc0];
      s1 = d.cell_start[cc0 + 1];
      s2 = m >= 1 ? d.cell_start[cc0 + 2] : s1;
      lo = s0;
      hi_end = d.cell_start[cc0 + m + 1];
      if (!exact_all) {
        const float gx = fmaxf(dcx < 0 ? oxi : (dcx > 0 ? csx - oxi : 0.f), 0.f);
        const float gy = fmaxf(dcy < 0 ? oyi : (dcy > 0 ? csy - oyi : 0.f), 0.f);
        const float rho2 = gx * gx + gy * gy;
        if (rho2 > ri2) {
          hi_end = lo;
        } else {
          const float w = sqrtf(ri2 - rho2);
          const int glo = min(max((int)floorf((bz0 - w) * inv_hz), 0), gmax);
          const int ghi = min(max((int)floorf((bz0 + w) * inv_hz), 0), gmax);
          const int alo = glo >> 2, klo = glo & 3, ahi = ghi >> 2, khi = ghi & 3;
          const int4 ol = d.soff[cc0 + alo], oh = d.soff[cc0 + ahi];
          lo = klo == 0 ? (alo == 0 ? s0 : (alo == 1 ? s1 : s2)) : (klo == 1 ? ol.x : (klo == 2 ? ol.y : ol.z));
          hi_end = khi == 3 ? oh.w : (khi == 0 ? oh.x : (khi == 1 ? oh.y : oh.z));
        }
      }
    }
  }
  int cnt = 0;
  for (int col = 0; col < 9; ++col) {
    const int p0 = __shfl(lo, seg + col, 64), p1 = __shfl(hi_end, seg + col, 64);
    const int q1 = __shfl(s1, seg + col, 64), q2 = __shfl(s2, seg + col, 64);
    const float cbx = __shfl(bx, seg + col, 64), cby = __shfl(by, seg + col, 64);
    // (the particles of a wavefront go round together)
    for (int base = 0; __any(p0 + base < p1); base += kBuildLanes) {
      const int p = p0 + base + sl;
      bool in = false;
      int j = 0;
      if (p < p1) {
        const int2 f = d.sinfo[p];
        const float4 q = d.sxyz[p];
        j = f.x;
        const float bz = p >= q2 ? bz2 : (p >= q1 ? bz1 : bz0);
        const float dx = cbx - q.x, dy = cby - q.y, dz = bz - q.z;
        const float r2 = dx * dx + dy * dy + dz * dz;
        const float t = hcf * (hi + q.w);
        const float t2 = t * t;
        const bool valid = (j != i) & (f.y == g);
        in = valid & (r2 < t2);
        if (valid & (exact_all | (fabsf(r2 - t2) <= 1e-4f * t2))) in = in_radius(xi, d.xh[cur][j], d.cellfac);
      }
      const unsigned mask = (unsigned)(__ballot(in) >> seg);
      const int k = cnt + __popc(mask & ((1u << sl) - 1u));
      if (in && k < d.max_nb) d.nbr[nb_slot(np, k, i)] = j;
      cnt += __popc(mask);
    }
  }
  if (i < d.n) {
    const int kept = cnt < d.max_nb ? cnt : d.max_nb;
    // the rest of the last group of four holds the particle itself
    if (sl < ((4 - (kept & 3)) & 3)) d.nbr[nb_slot(np, kept + sl, i)] = i;
    if (sl == 0) {
      d.nnb[i] = kept;
      if (cnt > d.max_nb) d.flags->overflow = 1;
    }
  }
  const double own = sl == 0 ? (double)cnt : 0.0;
  const double bt = block_reduce<0>(own, sh);
  const double bm = block_reduce<1>(own, sh);
  if (threadIdx.x == 0) {
    atomicAdd((unsigned long long *)&d.flags->directed_pairs, (unsigned long long)bt);
    atomicMax(&d.flags->max_count, (int)bm);
  }
}

// LDS staging lists of the pair passes, per tile of kBlock
// consecutive particles after every neighbour build: the tile's particles
// and all their neighbour entries go into an LDS hash set (open
// addressing); its distinct values (the staged set, ~6 % of the ~7000
// entries: each neighbour appears in many rows) are sorted (bitonic, in
// registers and lane shuffles) so a pass loads the set in long contiguous
// runs; each value's hash
// slot then records its position in the set, and every row entry is
// rewritten as that position.  The hash table's layout depends on insertion
// order, the sorted set does not.  Tiles whose set exceeds stage_max keep
// stage_cnt = -1 and gather from HBM.  Rows keep their order, so staged and
// HBM gathers sum in the same order.
constexpr int kStageThreads = 256;
constexpr int kHashSlots = 2048;  // >= 2 kStageMax: load <= 1/2 for sets of <= kStageMax values
static_assert(kHashSlots >= 2 * kStageMax && (kHashSlots & (kHashSlots - 1)) == 0, "hash table size");
static_assert(kStagePow2 >= kStageMax && (kStagePow2 & (kStagePow2 - 1)) == 0, "sort padding");
static_assert(kStageThreads == 2 * kBlock, "two threads per particle of a tile");
__device__ inline unsigned stage_hash(int v) { return ((unsigned)v * 2654435761u) >> 21; }  // 11 bits
static_assert(kStagePow2 == 4 * kStageThreads, "the set sort holds four values per thread");

// Bitonic sort (ascending) of the first P values (P a power of two <=
// kStagePow2) of the block, element e = 4 tid + r held in v[r]; elements at
// e >= P must hold values >= every value below P.  Compare-exchanges within
// a thread (j = 1, 2) stay in registers, those within a wavefront
// (4 <= j < 256) exchange through lane shuffles, and only j >= 256 goes
// through LDS (buf: kStagePow2 ints), two barriers each.  Every thread of
// the block calls this with the same P.
__device__ inline void stage_sort(int (&v)[4], int P, int *buf) {
  const int tid = threadIdx.x;
  for (int k = 2; k <= P; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      if (j >= 4) {
        int o[4];
        if (j >= 256) {
          reinterpret_cast<int4 *>(buf)[tid] = make_int4(v[0], v[1], v[2], v[3]);
          __syncthreads();
          const int4 w = reinterpret_cast<const int4 *>(buf)[tid ^ (j >> 2)];
          __syncthreads();
          o[0] = w.x;
          o[1] = w.y;
          o[2] = w.z;
          o[3] = w.w;
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = __shfl_xor(v[r], j >> 2, 64);
        }
        // the element at the lower index of its pair keeps the minimum when
        // the run (e & k) sorts ascending
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int e = 4 * tid + r;
          const bool keep_min = ((e & j) == 0) == ((e & k) == 0);
          v[r] = keep_min ? min(v[r], o[r]) : max(v[r], o[r]);
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (r & j) continue;
          const int e = 4 * tid + r;
          const int a = v[r], b = v[r ^ j];
          const bool asc = (e & k) == 0;
          v[r] = asc ? min(a, b) : max(a, b);
          v[r ^ j] = asc ? max(a, b) : min(a, b);
        }
      }
    }
  }
}

__global__ __launch_bounds__(kStageThreads) void k_stage(Dev d, int force) {
  if (!force && !d.flags->do_search) return;
  __shared__ int uniq[kStagePow2];
  __shared__ int ht[kHashSlots];
  __shared__ unsigned short hp[kHashSlots];
  __shared__ int nset, full;
  __shared__ int sh[34];
  const int tid = threadIdx.x, li = tid % kBlock, half = tid / kBlock;
  const long long np = d.npad;
  constexpr unsigned mask = kHashSlots - 1;
  for (int t = blockIdx.x; t < d.ntiles; t += gridDim.x) {
    const int i = t * kBlock + li;
    const int c = (i < d.n && d.group[i] >= 0) ? d.nnb[i] : 0;
    for (int p = tid; p < kHashSlots; p += kStageThreads) ht[p] = -1;
    if (tid == 0) {
      nset = 0;
      full = 0;
    }
    __syncthreads();
    // a value is counted by the thread whose CAS claims its slot; probing
    // stops once the set has more than stage_max values (the tile then
    // gathers from HBM), and every probe sequence ends within kHashSlots.
    // A group's four home-slot CAS are issued together (they are
    // independent; a lane's atomics on one slot apply in order, so the
    // repeated padding entries find their own value); only collisions
    // probe on, one value at a time.
    auto insert4 = [&](const int4 v4) {
      if (*(volatile int *)&full) return;
      const int vv[4] = {v4.x, v4.y, v4.z, v4.w};
      unsigned s[4];
      int old[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) s[u] = stage_hash(vv[u]) & mask;
#pragma unroll
      for (int u = 0; u < 4; ++u) old[u] = atomicCAS(&ht[s[u]], -1, vv[u]);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        int o = old[u];
        unsigned sl = s[u];
        for (int probe = 1; probe < kHashSlots && o != -1 && o != vv[u]; ++probe) {
          if (*(volatile int *)&full) break;
          sl = (sl + 1) & mask;
          o = atomicCAS(&ht[sl], -1, vv[u]);
        }
        if (o == -1 && atomicAdd(&nset, 1) >= d.stage_max) full = 1;
      }
    };
    // a row's groups of four entries (the last padded with i itself), the
    // two halves taking alternate groups, four groups' loads in flight; the
    // groups read past a row's end lie inside the row allocation
    const int4 *row = reinterpret_cast<const int4 *>(d.nbr) + i;
    const int ng = (c + 3) >> 2;
    if (i < d.n) {
      if (half == 0) insert4(make_int4(i, i, i, i));
      for (int g0 = half; g0 < ng; g0 += 8) {
        int4 v[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] = row[(long long)(g0 + 2 * b) * np];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          if (g0 + 2 * b >= ng) break;
          insert4(v[b]);
        }
      }
    }
    __syncthreads();
    if (full || nset > d.stage_max) {
      if (tid == 0) d.stage_cnt[t] = -1;
      __syncthreads();
      continue;
    }
    // compact the table: thread tid takes slots [8 tid, 8 tid + 8), one
    // block scan places its values (the order is irrelevant: sorted next)
    constexpr int kSlotsPer = kHashSlots / kStageThreads;
    static_assert(kSlotsPer == 8, "two int4 loads of slots per thread");
    const int4 h0 = reinterpret_cast<const int4 *>(ht)[2 * tid];
    const int4 h1 = reinterpret_cast<const int4 *>(ht)[2 * tid + 1];
    const int hv[8] = {h0.x, h0.y, h0.z, h0.w, h1.x, h1.y, h1.z, h1.w};
    int f = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) f += hv[q] >= 0 ? 1 : 0;
    int U;
    int e = block_scan_excl(f, sh, &U);
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (hv[q] >= 0) uniq[e++] = hv[q];
    int P = 1;
    while (P < U) P <<= 1;
    __syncthreads();
    int sv[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) sv[r] = 4 * tid + r < U ? uniq[4 * tid + r] : 0x7fffffff;
    __syncthreads();
    stage_sort(sv, P, uniq);
    // each value's slot records its position in the sorted set
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int p = 4 * tid + r;
      if (p < U) {
        const int v = sv[r];
        unsigned s = stage_hash(v) & mask;
        while (ht[s] != v) s = (s + 1) & mask;
        hp[s] = (unsigned short)p;
        d.stage[(long long)t * kStageMax + p] = v;
      }
    }
    __syncthreads();
    auto pos = [&](int v) -> unsigned short {
      unsigned s = stage_hash(v) & mask;
      while (ht[s] != v) s = (s + 1) & mask;
      return hp[s];
    };
    if (i < d.n) {
      if (half == 0) d.selfl[i] = pos(i);
      // the padding entries hold i, so they become the particle's own position
      ushort4 *rowl = reinterpret_cast<ushort4 *>(d.nbrl) + i;
      for (int g0 = half; g0 < ng; g0 += 8) {
        int4 v[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] = row[(long long)(g0 + 2 * b) * np];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          if (g0 + 2 * b >= ng) break;
          rowl[(long long)(g0 + 2 * b) * np] = make_ushort4(pos(v[b].x), pos(v[b].y), pos(v[b].z), pos(v[b].w));
        }
      }
    }
    if (tid == 0) d.stage_cnt[t] = U;
    __syncthreads();
  }
}

// Domain::CalcGradCorrMatrix (Source/Domain.cpp:1832-1940):
// L_i = (-sum_j V_j GK_ij x_ij (x) x_ij)^-1 over i's neighbour row (FP64
// gather, V_j = m_j / rho_j, x_ij = x_i - x_j; in 2D the sum's zz entry is
// set to 1 before the inversion), symmetric; the identity
// where |det| < 1e-10 (InvLog, External/matvec.h:673-693) and for fixed
// particles.  Runs when the schedule set gc_due.
WF_KERNEL void k_gradcorr(Dev d, int cur) {
  if (!d.flags->gc_due) return;
  const long long np = d.npad;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < d.n; i += gridDim.x * kBlock) {
    double L[6] = {1.0, 1.0, 1.0, 0.0, 0.0, 0.0};
    if (d.group[i] >= 0) {
      const double4 xi = d.xh[cur][i];
      const KH<double> ki = kern_h_t<double>(xi.w, d.dim);
      double m[6] = {0, 0, 0, 0, 0, 0};
      const int cnt = d.nnb[i];
      for (int k = 0; k < cnt; ++k) {
        const int j = d.nbr[nb_slot(np, k, i)];
        const double4 xj = d.xh[cur][j];
        const double dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
        const double GK = gk_t<double>(dx * dx + dy * dy + dz * dz, pair_h_t<double>(ki, xi.w, xj.w));
        const double w = d.vol[cur][j] * GK;
        m[XX] -= w * dx * dx;
        m[YY] -= w * dy * dy;
        m[ZZ] -= w * dz * dz;
        m[XY] -= w * dx * dy;
        m[XZ] -= w * dx * dz;
        m[YZ] -= w * dy * dz;
      }
      if (d.dim == 2) m[ZZ] = 1.0;  // the 2D sum's zz entry (Source/Domain.cpp:1911-1915)
      const double c00 = m[YY] * m[ZZ] - m[YZ] * m[YZ], c01 = m[XZ] * m[YZ] - m[XY] * m[ZZ];
      const double c02 = m[XY] * m[YZ] - m[XZ] * m[YY];
      const double det = m[XX] * c00 + m[XY] * c01 + m[XZ] * c02;
      if (fabs(det) >= 1.0e-10) {
        L[XX] = c00 / det;
        L[XY] = c01 / det;
        L[XZ] = c02 / det;
        L[YY] = (m[XX] * m[ZZ] - m[XZ] * m[XZ]) / det;
        L[YZ] = (m[XZ] * m[XY] - m[XX] * m[YZ]) / det;
        L[ZZ] = (m[XX] * m[YY] - m[XY] * m[XY]) / det;
      }
    }
    for (int k = 0; k < 6; ++k) d.gcm[k * np + i] = L[k];
  }
}

void launch_gradcorr(const Dev &d, hipStream_t st, int cur) {
  k_gradcorr<<<nblk_small(d.n), kBlock, 0, st>>>(d, cur);
}

// plane strain: StartAcceleration resets each particle's z velocity at the
// top of every step (Source/Domain.cpp:1592); the FP32 shadow with it
WF_KERNEL void k_plane_strain(Dev d) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= d.n) return;
  d.vm[i].z = 0.0;
  if (d.mixed) d.vmf[i].z = 0.0f;
}
void launch_plane_strain(const Dev &d, hipStream_t st) { k_plane_strain<<<d.nblocks, kBlock, 0, st>>>(d); }

void launch_schedule(const Dev &d, hipStream_t st, int force, const BcTable *bc) {
  const int rigid = bc && d.contact;
  k_schedule<<<rigid ? nblk(d.nrig) : 1, kBlock, 0, st>>>(d, force, rigid, bc ? *bc : BcTable{});
}

// rows built with kBuildLanes lanes per particle up to this many particles: the
// whole search with 32 lanes against one 94 and 139 us at 1.3k, 107 and 138 at
// 3.1k, 131 and 148 at 6.2k, 143 and 153 at 7.7k, and slower at 35k.  Plane
// strain has a third of the candidates, for which 32 lanes are mostly idle: 67
// and 78 us at 1.1k, 73 and 77 at 2.1k, but 88 and 77 at 4.6k, 110 and 77 at 8.1k.
constexpr int kBuildWide = 8192, kBuildWide2d = 2048;
void launch_neighbours(const Dev &d, hipStream_t st, int cur) {
  k_cell_hist<<<nblk((long long)d.n + d.nrig), kBlock, 0, st>>>(d, cur);
  k_scan<<<scan_chunks(d.sncells) + (d.nrig ? scan_chunks(d.ncells) : 0), kScanThreads, 0, st>>>(d);
  k_scatter<<<nblk((long long)d.n + d.nrig), kBlock, 0, st>>>(d);
  // (at most 8192 blocks: an idle launch of that size costs about as much
  // as the other search kernels', and 16k wavefronts keep the cells' loads
  // in flight)
  {
    const int waves = kSortBlocks * (kBlock / 64);
    int group = (d.sncells + waves - 1) / waves;
    group = group < kSortGroup ? group : kSortGroup;
    const int g = nblk((long long)(d.sncells + group - 1) / group * 64);
    k_cell_sort<<<g < kSortBlocks ? g : kSortBlocks, kBlock, 0, st>>>(d, cur, group);
  }
  if (d.n <= (d.dim == 2 ? kBuildWide2d : kBuildWide)) k_build_nbr_wide<<<nblk((long long)d.n * kBuildLanes), kBlock, 0, st>>>(d, cur);
  else k_build_nbr<<<nblk(d.n), kBlock, 0, st>>>(d, cur);
  if (d.stage_max > 0) k_stage<<<d.ntiles < 2048 ? d.ntiles : 2048, kStageThreads, 0, st>>>(d, 0);
}
void launch_stage(const Dev &d, hipStream_t st) {
  if (d.stage_max > 0) k_stage<<<d.ntiles < 2048 ? d.ntiles : 2048, kStageThreads, 0, st>>>(d, 1);
}

// ---------------------------------------------------------------------------
// pass 1: acceleration (CalcAccel + AccelReduction, GradientType 0, TI = 0)

// P / rho^2 with the equation of state's P.  Rounded here, not fused into the
// sum that takes it: a neighbour's value is the same from HBM and from LDS
__device__ inline double pr_of(double rho, double P0, double cs2, double rho0) {
#pragma clang fp contract(off)
  const double ir = rcp_t(rho);
  return (P0 + cs2 * (rho - rho0)) * ir * ir;
}

// Where a pass reads neighbour j: straight from HBM (Src<MX>, row of global
// indices in nbr) or from the tile's LDS copy (row of staged positions in
// nbrl).  Both give the same values, so results do not depend on staging.
template <bool MX>
struct HbmJ {
  using S = Src<MX>;
  using R = typename S::R;
  using R4 = typename S::R4;
  // FP64 gathers: a batch of 4 in flight (8 costs more registers than it
  // gains); FP32: the whole batch
  static constexpr int kUnroll = MX ? kNbBatch : 4;
  const Dev &d;
  const int buf;
  const int i;
  // entries k0..k0+7 (k0 a multiple of 8) of particle i's row
  __device__ void fetch(int k0, int out[kNbBatch]) const {
    const int4 *row = reinterpret_cast<const int4 *>(d.nbr) + i;
    const int4 a = row[(long long)(k0 >> 2) * d.npad];
    const int4 b = row[(long long)((k0 >> 2) + 1) * d.npad];
    out[0] = a.x, out[1] = a.y, out[2] = a.z, out[3] = a.w;
    out[4] = b.x, out[5] = b.y, out[6] = b.z, out[7] = b.w;
  }
  __device__ int self() const { return i; }
  __device__ R4 x(int j) const { return S::x(d, buf, j); }
  __device__ R4 v(int j) const { return S::v(d, j); }
  __device__ void srec(int j, R t[6], R &rho) const { S::srec(d, j, t, rho); }
  // tensile-instability stress of particle j
  __device__ void tir(int j, R t[6]) const {
    for (int k = 0; k < 6; ++k) {
      if constexpr (MX) t[k] = d.tirf[(long long)k * d.npad + j];
      else t[k] = d.tir[(long long)k * d.npad + j];
    }
  }
  // m_j / rho_j and, with damage, the damage of particle j (FP64 passes)
  __device__ R vol(int j) const { return S::vol(d, buf, j, R4{}); }
  __device__ R dam(int j) const { return d.damD[j]; }
  // P_j / rho_j^2 of the kinetic-energy pair term (FP64 passes)
  __device__ R pr(int j, R P0, R cs2, R rho0) const { return pr_of(d.rho[buf][j], P0, cs2, rho0); }
  __device__ bool lower(int j) const { return i < j; }
};

// Calls f(j) for the entries of a neighbour row of cnt entries that belong
// to lane `sub` of the particle's `lanes` lanes: batches of kNbBatch entries
// sub, sub + lanes, sub + 2 lanes, ... in row order, each batch's indices
// fetched while the previous batch is processed.  Entries past cnt in the
// last batch call f with j = the particle itself: a particle paired with
// itself has x_ij = v_ij = 0, so every pair term is an exact zero and adding
// it changes no sum.
template <class G, class F>
__device__ inline void for_each_nb(const G &g, int cnt, int sub, int lanes, F &&f) {
  int cur[kNbBatch], nxt[kNbBatch];
  const int step = lanes * kNbBatch;
  int base = sub * kNbBatch;
  g.fetch(base, cur);
  const int self = g.self();
  for (; base < cnt; base += step) {
    g.fetch(base + step, nxt);
#pragma unroll G::kUnroll
    for (int u = 0; u < kNbBatch; ++u) f(base + u < cnt ? cur[u] : self);
#pragma unroll
    for (int u = 0; u < kNbBatch; ++u) cur[u] = nxt[u];
  }
}

// copy the tile's staged set into LDS (all NT threads of the block call
// these).  A thread's share (entries p = tid + r NT) is loaded in three
// rounds, each with all of the share's loads in flight: the set's particle
// indices, then the records (from particle 0 for entries past the set's
// end, so no load is conditional), then the LDS stores of the set's
// entries.  Entries past the set's end are stored to the spare slot
// kStageMax (the LDS arrays hold kStageMax + 1 records), so no store is
// conditional either and nothing moves a load down to its store.
// density / rates: (x, m/rho), (v, m) and, for rates, P / rho^2
template <int NT>
__device__ inline void stage_xv(const Dev &d, int t, int U, const float4 *gx, float4 *lx, float4 *lv, float *lp) {
  constexpr int R = (kStageMax + NT - 1) / NT;
  const int *st = d.stage + (long long)t * kStageMax;
  int j[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int p = (int)threadIdx.x + r * NT;
    j[r] = p < U ? st[p] : 0;
  }
  float4 x[R], v[R];
  float pr[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    x[r] = gx[j[r]];
    v[r] = d.vmf[j[r]];
    if (lp) pr[r] = d.prf[j[r]];
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int p = (int)threadIdx.x + r * NT;
    const int q = p < U ? p : kStageMax;
    lx[q] = x[r];
    lv[q] = v[r];
    if (lp) lp[q] = pr[r];
  }
  __syncthreads();
}
// acceleration: (x, rho), (v, m), sigma / rho^2 as (t0..t3), (t4, t5)
template <int NT>
__device__ inline void stage_accel(const Dev &d, int t, int U, const float4 *gx, float4 *lx, float4 *lv, float4 *lt,
                                   float2 *lt2) {
  constexpr int R = (kStageMax + NT - 1) / NT;
  const int *st = d.stage + (long long)t * kStageMax;
  const float4 *gs = reinterpret_cast<const float4 *>(d.srecf);  // (t0..t3), (t4, t5, rho, pad)
  int j[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int p = (int)threadIdx.x + r * NT;
    j[r] = p < U ? st[p] : 0;
  }
  float4 x[R], v[R], s0[R], s1[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    x[r] = gx[j[r]];
    v[r] = d.vmf[j[r]];
    s0[r] = gs[2 * j[r]];
    s1[r] = gs[2 * j[r] + 1];
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int p = (int)threadIdx.x + r * NT;
    const int q = p < U ? p : kStageMax;
    lx[q] = make_float4(x[r].x, x[r].y, x[r].z, s1[r].z);
    lv[q] = v[r];
    lt[q] = s0[r];
    lt2[q] = make_float2(s1[r].x, s1[r].y);
  }
  __syncthreads();
}

// cubic-spline kernel shape w(q) = W(q h) pi h^3 (Source/Functions.cpp:25-37)
template <typename R>
__device__ inline R w_shape(R q) {
  const R t = (R)2 - q;
  return q < (R)1 ? (R)1 - (R)1.5 * q * q + (R)0.75 * q * q * q : (q < (R)2 ? (R)0.25 * t * t * t : (R)0);
}

// TI: with the tensile-instability term (W(r)/W(d0))^n (TIR_i + TIR_j) of
// CalcAccel (Source/InteractionAlt.cpp:104-110); pairs form within one
// material, so n and d0 are the material's
// particle i's gradCorrM (symmetric, 6 components): the identity when the
// correction is off
template <bool GC, typename R>
__device__ inline void own_corr(const Dev &d, int i, R (&L)[6]) {
  L[XX] = L[YY] = L[ZZ] = (R)1;
  L[XY] = L[XZ] = L[YZ] = (R)0;
  if constexpr (GC)
    for (int k = 0; k < 6; ++k) L[k] = (R)d.gcm[(long long)k * d.npad + i];
}
// e = L x_ij: the direction the kernel gradient GK e takes under the
// correction, (GK L) x_ij of Source/InteractionAlt.cpp:118-133
template <bool GC, typename R>
__device__ inline void corr_dir(const R (&L)[6], R dx, R dy, R dz, R &ex, R &ey, R &ez) {
  if constexpr (GC) {
    ex = L[XX] * dx + L[XY] * dy + L[XZ] * dz;
    ey = L[XY] * dx + L[YY] * dy + L[YZ] * dz;
    ez = L[XZ] * dx + L[YZ] * dy + L[ZZ] * dz;
  } else {
    ex = dx, ey = dy, ez = dz;
  }
}

// GC: with the kernel-gradient correction (particle i's own gradCorrM
// applied to x_ij in the pair term)
template <bool MX, bool TI, bool GC, class G>
__device__ inline void accel_lane(const Dev &d, int cur, int i, const G &g, int sub, int lanes,
                                  typename Src<MX>::R (&acc)[3]) {
  using S = Src<MX>;
  using R = typename S::R;
  R ax = 0, ay = 0, az = 0;
  if (d.group[i] >= 0) {
    R Li[6];
    own_corr<GC>(d, i, Li);
    const DevMat &M = d.mats[d.mat[i]];
    const R alpha = (R)M.alpha, beta = (R)M.beta, cs = (R)M.Cs;
    const bool av = (M.alpha != 0.0 || M.beta != 0.0);
    const auto xi = S::x(d, cur, i);
    const auto vi = S::v(d, i);
    R ti[6], rhoi;
    S::srec(d, i, ti, rhoi);
    const KH<R> ki = kern_h_t<R>(S::h_own(d, cur, i, xi), d.dim);
    const R acs = alpha * cs;
    R tri[6] = {0, 0, 0, 0, 0, 0};
    const R tin = (R)M.ti_n, tid = (R)M.ti_dist;
    if constexpr (TI) g.tir(i, tri);
    for_each_nb(g, d.nnb[i], sub, lanes, [&](int j) {
      const auto xj = g.x(j);
      const auto vj = g.v(j);
      R tj[6], rhoj;
      g.srec(j, tj, rhoj);
      const KH<R> kh = S::kh(ki, xi, xj);
      const R dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
      const R r2 = dx * dx + dy * dy + dz * dz;
      const R GK = gk_t<R>(r2, kh);
      // Monaghan viscosity for approaching pairs (selected, not branched):
      // mu = h vdot / D1, Pi = mu (alpha cs + beta mu) / D2 with a single
      // reciprocal of D1 D2 (D1 = r^2 + 0.01 h^2, D2 = (rho_i + rho_j) / 2)
      const R vdot = (vi.x - vj.x) * dx + (vi.y - vj.y) * dy + (vi.z - vj.z) * dz;
      const R D1 = r2 + (R)0.01 * kh.h * kh.h, D2 = (R)0.5 * (rhoi + rhoj);
      const R hv = kh.h * vdot * rcp_t(D1 * D2);
      const R pv = hv * (acs + beta * (hv * D2));
      const R pi = (av && vdot < (R)0) ? pv : (R)0;
      const R Mxx = ti[XX] + tj[XX] + pi;
      const R Myy = ti[YY] + tj[YY] + pi;
      const R Mzz = ti[ZZ] + tj[ZZ] + pi;
      R Mxy = ti[XY] + tj[XY];
      R Mxz = ti[XZ] + tj[XZ];
      R Myz = ti[YZ] + tj[YZ];
      R Mxx2 = Mxx, Myy2 = Myy, Mzz2 = Mzz;
      if constexpr (TI) {
        // a padded self entry has r2 = 0: q = 0 keeps the factor finite
        const R q = r2 > (R)0 ? r2 * rsqrt_t(r2) * kh.ih : (R)0;
        const R s = pow(w_shape<R>(q) / w_shape<R>(tid * kh.ih), tin);
        R trj[6];
        g.tir(j, trj);
        Mxx2 += s * (tri[XX] + trj[XX]);
        Myy2 += s * (tri[YY] + trj[YY]);
        Mzz2 += s * (tri[ZZ] + trj[ZZ]);
        Mxy += s * (tri[XY] + trj[XY]);
        Mxz += s * (tri[XZ] + trj[XZ]);
        Myz += s * (tri[YZ] + trj[YZ]);
      }
      R w = vj.w * GK;
      if constexpr (!MX) {
        // damage weight of the pair (Source/InteractionAlt.cpp:54-60)
        if (d.damage) {
          const R df = dam_weight(d.damD[i], g.dam(j));
          w = df > (R)0 ? (df * vj.w) * GK : (R)0;
        }
      }
      R ex, ey, ez;
      corr_dir<GC>(Li, dx, dy, dz, ex, ey, ez);
      ax += w * (ex * Mxx2 + ey * Mxy + ez * Mxz);
      ay += w * (ex * Mxy + ey * Myy2 + ez * Myz);
      az += w * (ex * Mxz + ey * Myz + ez * Mzz2);
    });
  }
  acc[0] = ax;
  acc[1] = ay;
  acc[2] = az;
}

// ---------------------------------------------------------------------------
// Mixed-precision pair passes (no tensile instability).  A lane walks its
// particle's row in groups of four entries (rows are padded to a multiple
// of four with the particle itself, whose pair terms are exact zeros):
// lane `sub` of LANES takes groups sub, sub + LANES, ..., the row words two
// groups ahead in flight.  All four neighbours' records of a group are
// loaded before any is used and the pair arithmetic has no branch, so a
// group's loads are in flight together.  The records come from the tile's
// LDS copy (row entries are positions in the staged set, nbrl) or, for a
// tile whose set did not fit, straight from HBM (row entries are particle
// indices, nbr); both give the same values in the same order.

// particle i's kernel constants for the FP32 gradient factor
struct GkF {
  float ih, gin_a, gin_b, gout;  // 1/h, 2.25 c5, -3 c5, -0.75 c5 h
};
__device__ inline GkF gk_consts(float h, int dim) {
  const KH<float> k = kern_h_t<float>(h, dim);
  return GkF{k.ih, 2.25f * k.c5, -3.0f * k.c5, -0.75f * k.c5 * h};
}
// GK of the cubic spline (Source/Functions.cpp:74-87) for r2 = |x_ij|^2:
// c5 (2.25 q - 3) for q < 1, -0.75 c5 h (2 - q)^2 / r for 1 <= q < 2, 0
// beyond, selected without a branch.  r2 = 0 (a padded self entry, or two
// coincident particles) gives q = 0 and GK = -3 c5, the reference's q = 0
// value, with every operand finite.
__device__ inline float gk_f(float r2, const GkF &k) {
  const float ri = __builtin_amdgcn_rsqf(fmaxf(r2, FLT_MIN));
  const float q = (r2 * ri) * k.ih;
  const float gin = fmaf(q, k.gin_a, k.gin_b);
  const float t = fmaxf(2.0f - q, 0.0f);
  const float gout = (t * t) * (ri * k.gout);
  return q < 1.0f ? gin : gout;
}

// ---------------------------------------------------------------------------
// FP64 pair passes from the tile's LDS copy, for contexts whose smoothing
// length is uniform within each material (h_uni; the HBM gathers further down
// cover the others).  The same rows, walk and branch-free pair arithmetic as
// the mixed passes, in double.  LANES threads per particle; a tile that is
// not staged reads the same records from HBM, in the same order.
//
// The HBM gathers are bound by the L1 and L2 traffic of 128 (acceleration),
// 72 and 80 bytes per neighbour; the LDS copy is read from HBM once per tile
// (~730 records for 128 particles), which leaves FP64 issue and LDS reads (112
// bytes per pair in the acceleration) as the bounds.  Acceleration, density,
// rates per launch at 976k particles (54.6 neighbours): gathers 735, 426 and
// 480 us, from LDS 318, 146 and 191 us; at 4.5k particles 21.8, 16.1 and
// 20.7 against 10.6, 7.3 and 9.5 us.
//
// A compile-time option (GC, BETA, DAM) costs no registers where it is off:
// a runtime `if (damage)` in the walk split it into blocks and spilled 489
// registers.

// gk_f in double
__device__ inline double gk_d(double r2, const GkD &k) {
  const double ri = rsqrt3(fmax(r2, DBL_MIN));
  const double q = (r2 * ri) * k.ih;
  const double gin = fma(q, k.gin_a, k.gin_b);
  const double t = fmax(2.0 - q, 0.0);
  const double gout = (t * t) * (ri * k.gout);
  return q < 1.0 ? gin : gout;
}

// A tile's records in LDS, as arrays of 16-byte pairs: 16-byte reads of
// consecutive positions cover every bank (32-byte records would use half of
// them per read).  (x, y), (z, w), (vx, vy), (vz, u) with w and u = rho and m
// (acceleration) or m/rho and m (rates); density: (x, y), (z, m/rho),
// (vx, vy) and vz alone.  The acceleration adds sigma / rho^2 as three pairs.
constexpr int kRecAccel = 7, kRecRates = 4, kRecDens = 3;  // pairs per record
enum { PASS_ACCEL, PASS_DENS, PASS_RATES };
template <int PASS>
struct RecLds64 {
  const double2 *r;
  const double *s;   // vz (density), P/rho^2 (rates)
  const double *dm;  // damage
  __device__ void x(int p, double &x, double &y, double &z, double &w) const {
    const double2 a = r[p], b = r[kStageMax + p];
    x = a.x, y = a.y, z = b.x, w = b.y;
  }
  __device__ void v(int p, double &x, double &y, double &z, double &u) const {
    const double2 a = r[2 * kStageMax + p];
    x = a.x, y = a.y;
    if constexpr (PASS == PASS_DENS) {
      z = s[p], u = 0.0;
    } else {
      const double2 b = r[3 * kStageMax + p];
      z = b.x, u = b.y;
    }
  }
  __device__ void t(int p, double (&t)[6]) const {
    const double2 a = r[4 * kStageMax + p], b = r[5 * kStageMax + p], c = r[6 * kStageMax + p];
    t[0] = a.x, t[1] = a.y, t[2] = b.x, t[3] = b.y, t[4] = c.x, t[5] = c.y;
  }
  __device__ double pr(int p) const { return s[p]; }
  __device__ double dam(int p) const { return dm[p]; }
};
template <int PASS>
struct RecHbm64 {
  const Dev &d;
  const int buf;
  __device__ void x(int j, double &x, double &y, double &z, double &w) const {
    const double4 a = d.xh[buf][j];
    x = a.x, y = a.y, z = a.z;
    if (PASS == PASS_ACCEL) w = d.srec[j].rho;
    else w = rec_vol(d, buf, j, PASS == PASS_RATES);
  }
  __device__ void v(int j, double &x, double &y, double &z, double &u) const {
    const double4 a = d.vm[j];
    x = a.x, y = a.y, z = a.z, u = a.w;
  }
  __device__ void t(int j, double (&t)[6]) const {
    const StressRec q = d.srec[j];
    for (int k = 0; k < 6; ++k) t[k] = q.s[k] * q.irho2;
  }
  __device__ double pr(int j) const { return rec_pr(d, buf, j); }
  __device__ double dam(int j) const { return d.damD[j]; }
  // m / rho, rounded to float in the rates of the Locking sums
  __device__ static double rec_vol(const Dev &d, int buf, int j, bool rates) {
    const double w = d.vol[buf][j];
    return rates && d.locking ? (double)(float)w : w;
  }
  // P / rho^2 of the equation of state (pairs form within one material, so
  // j's own material is the pair's)
  __device__ static double rec_pr(const Dev &d, int buf, int j) {
    const DevMat &M = d.mats[d.mat[j]];
    return pr_of(d.rho[buf][j], M.P0, M.Cs * M.Cs, M.ref_density);
  }
};
template <int NT, int PASS>
__device__ inline void stage64(const Dev &d, int buf, int t, int U, double2 *r, double *sc, double *dm) {
  const RecHbm64<PASS> h{d, buf};
  stage_set<NT>(d.stage, t, U, [&](int p, int j) {
    double x, y, z, w, vx, vy, vz, u;
    h.x(j, x, y, z, w);
    h.v(j, vx, vy, vz, u);
    if constexpr (PASS == PASS_ACCEL) {
      double s[6];
      h.t(j, s);
      r[4 * kStageMax + p] = make_double2(s[0], s[1]);
      r[5 * kStageMax + p] = make_double2(s[2], s[3]);
      r[6 * kStageMax + p] = make_double2(s[4], s[5]);
    }
    if constexpr (PASS == PASS_RATES) sc[p] = h.pr(j);
    r[p] = make_double2(x, y);
    r[kStageMax + p] = make_double2(z, w);
    r[2 * kStageMax + p] = make_double2(vx, vy);
    if constexpr (PASS == PASS_DENS) sc[p] = vz;
    else r[3 * kStageMax + p] = make_double2(vz, u);
    if constexpr (PASS != PASS_RATES)
      if (d.damage) dm[p] = h.dam(j);
  });
}

// CalcAccel + AccelReduction (Source/InteractionAlt.cpp:12-260), as
// accel_mx_lane in double, with the damage weight of the pair (:54-60)
template <bool GC, bool BETA, bool DAM, class Rows, class Rec>
__device__ inline void accel64_lane(const Dev &d, int i, int sub, int cnt, const double4 &xi, const double4 &vi,
                                    const StressRec &ri, const Rows &rows, typename Rows::G a0, typename Rows::G b0,
                                    const Rec &rec, double (&acc)[3]) {
  double ax = 0, ay = 0, az = 0, sx = 0, sy = 0, sz = 0;
  double Li[6];
  own_corr<GC>(d, i, Li);
  const DevMat &M = d.mats[d.mat[i]];
  const double h = xi.w, rhoi = ri.rho;
  const GkD k = gk_consts64(h, d.dim);
  const double h2c = 0.01 * h * h, acs = M.alpha * M.Cs, bh = 0.5 * M.beta, hh = 2.0 * h, hha = hh * acs;
  const double Di = DAM ? d.damD[i] : 0.0;
  walk_groups<kLanesLds64>(rows, cnt, sub, rows.self(), a0, b0, [&](const typename Rows::G &c) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int p = entry(c, u);
      double x, y, z, rho, vx, vy, vz, m, T[6];
      rec.x(p, x, y, z, rho);
      rec.v(p, vx, vy, vz, m);
      rec.t(p, T);
      const double dx = xi.x - x, dy = xi.y - y, dz = xi.z - z;
      const double r2 = dx * dx + dy * dy + dz * dz;
      const double GK = gk_d(r2, k);
      const double vdot = (vi.x - vx) * dx + (vi.y - vy) * dy + (vi.z - vz) * dz;
      const double D = rhoi + rho;
      const double rd = rcp3((r2 + h2c) * D);
      double pv;
      if constexpr (BETA) {
        const double hv = (hh * vdot) * rd;
        pv = hv * fma(bh, hv * D, acs);
      } else {
        pv = (hha * vdot) * rd;
      }
      const double pi = vdot < 0.0 ? pv : 0.0;
      double w = m * GK;
      if constexpr (DAM) {
        const double df = dam_weight(Di, rec.dam(p));
        w = df > 0.0 ? (df * m) * GK : 0.0;
      }
      double ex, ey, ez;
      corr_dir<GC>(Li, dx, dy, dz, ex, ey, ez);
      ax = fma(w, fma(T[XX], ex, fma(T[XY], ey, fma(T[XZ], ez, pi * ex))), ax);
      ay = fma(w, fma(T[XY], ex, fma(T[YY], ey, fma(T[YZ], ez, pi * ey))), ay);
      az = fma(w, fma(T[XZ], ex, fma(T[YZ], ey, fma(T[ZZ], ez, pi * ez))), az);
      sx = fma(w, ex, sx);
      sy = fma(w, ey, sy);
      sz = fma(w, ez, sz);
      // at most two entries' records in registers
      if (u & 1) __builtin_amdgcn_sched_barrier(0);
    }
  });
  double t[6];
  for (int q = 0; q < 6; ++q) t[q] = ri.s[q] * ri.irho2;
  acc[0] = ax + (t[XX] * sx + t[XY] * sy + t[XZ] * sz);
  acc[1] = ay + (t[XY] * sx + t[YY] * sy + t[YZ] * sz);
  acc[2] = az + (t[XZ] * sx + t[YZ] * sy + t[ZZ] * sz);
}

// CalcDensInc + DensReduction (Source/InteractionAlt.cpp:483-640) with the
// damage weight (:558-572)
template <bool GC, bool DAM, class Rows, class Rec>
__device__ inline double dens64_lane(const Dev &d, int i, int sub, int cnt, const double4 &xi, const double4 &vi,
                                     const Rows &rows, typename Rows::G a0, typename Rows::G b0, const Rec &rec) {
  double s = 0;
  double Li[6];
  own_corr<GC>(d, i, Li);
  const GkD k = gk_consts64(xi.w, d.dim);
  const double Di = DAM ? d.damD[i] : 0.0;
  walk_groups<kLanesLds64>(rows, cnt, sub, rows.self(), a0, b0, [&](const typename Rows::G &c) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int p = entry(c, u);
      double x, y, z, vol, vx, vy, vz, unused;
      rec.x(p, x, y, z, vol);
      rec.v(p, vx, vy, vz, unused);
      const double dx = xi.x - x, dy = xi.y - y, dz = xi.z - z;
      const double GK = gk_d(dx * dx + dy * dy + dz * dz, k);
      double ex, ey, ez;
      corr_dir<GC>(Li, dx, dy, dz, ex, ey, ez);
      const double t = (vi.x - vx) * ex + (vi.y - vy) * ey + (vi.z - vz) * ez;
      if constexpr (DAM) {
        const double df = dam_weight(Di, rec.dam(p));
        vol = df > 0.0 ? df * vol : 0.0;
      }
      s = fma(vol * GK, t, s);
      if (u & 1) __builtin_amdgcn_sched_barrier(0);
    }
  });
  return s;
}

// CalcRateTensors + RateTensorsReduction with the kinetic-energy pair term,
// as rates_mx_lane in double; own is the particle's entry in its own row
// (staged position or index)
template <bool GC, class Rows, class Rec>
__device__ inline void rates64_lane(const Dev &d, int i, int own, int sub, int cnt, const double4 &xi, const double4 &vi,
                                    double pri, const Rows &rows, typename Rows::G a0, typename Rows::G b0,
                                    const Rec &rec, double (&v)[10]) {
  double dxx = 0, dyy = 0, dzz = 0, pxy = 0, qxy = 0, pxz = 0, qxz = 0, pyz = 0, qyz = 0, ek = 0;
  double Li[6];
  own_corr<GC>(d, i, Li);
  const double mneg = -vi.w;
  const GkD k = gk_consts64(xi.w, d.dim);
  walk_groups<kLanesLds64>(rows, cnt, sub, rows.self(), a0, b0, [&](const typename Rows::G &c) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int p = entry(c, u);
      double x, y, z, vol, ux, uy, uz, m;
      rec.x(p, x, y, z, vol);
      rec.v(p, ux, uy, uz, m);
      const double pr = rec.pr(p);
      const double dx = xi.x - x, dy = xi.y - y, dz = xi.z - z;
      const double GK = gk_d(dx * dx + dy * dy + dz * dz, k);
      const double vx = vi.x - ux, vy = vi.y - uy, vz = vi.z - uz;
      const double cj = vol * GK;
      double ex, ey, ez;
      corr_dir<GC>(Li, dx, dy, dz, ex, ey, ez);
      const double a = cj * ex, b = cj * ey, g = cj * ez;
      dxx = fma(vx, a, dxx);
      dyy = fma(vy, b, dyy);
      dzz = fma(vz, g, dzz);
      pxy = fma(vx, b, pxy);
      qxy = fma(vy, a, qxy);
      pxz = fma(vx, g, pxz);
      qxz = fma(vz, a, qxz);
      pyz = fma(vy, g, pyz);
      qyz = fma(vz, b, qyz);
      // staged positions follow particle index order
      const double ms = own < p ? m : mneg;
      ek = fma(ms * (pri + pr), GK * (vx * dx + vy * dy + vz * dz), ek);
      if (u & 1) __builtin_amdgcn_sched_barrier(0);
    }
  });
  v[XX] = -dxx;
  v[YY] = -dyy;
  v[ZZ] = -dzz;
  v[XY] = -0.5 * (pxy + qxy);
  v[XZ] = -0.5 * (pxz + qxz);
  v[YZ] = -0.5 * (pyz + qyz);
  v[6] = -0.5 * (pxy - qxy);
  v[7] = -0.5 * (pxz - qxz);
  v[8] = -0.5 * (pyz - qyz);
  v[9] = 0.5 * ek;
}

// acceleration records of neighbour j: X = (x, y, z, rho), V = (v, m),
// T = sigma / rho^2 as (xx, yy, zz, xy), T2 = (xz, yz)
struct AccelLds {
  const float4 *lx, *lv, *lt;
  const float2 *lt2;
  __device__ void load(int l, float4 &X, float4 &V, float4 &T, float2 &T2) const {
    X = lx[l];
    V = lv[l];
    T = lt[l];
    T2 = lt2[l];
  }
};
struct AccelHbm {
  const float4 *gx, *gv;
  const float4 *gs;  // StressRecF as two float4: (t0..t3), (t4, t5, rho, pad)
  __device__ void load(int j, float4 &X, float4 &V, float4 &T, float2 &T2) const {
    const float4 x = gx[j], s1 = gs[2 * j + 1];
    V = gv[j];
    T = gs[2 * j];
    X = make_float4(x.x, x.y, x.z, s1.z);
    T2 = make_float2(s1.x, s1.y);
  }
};

// CalcAccel + AccelReduction in FP32 (Source/InteractionAlt.cpp:12-260,
// GradientType 0): a_i = sum_j m_j GK (sigma_i/rho_i^2 + sigma_j/rho_j^2 +
// Pi_ij) e_ij with e = x_ij (or gradCorrM_i x_ij).  The particle's own term
// sigma_i/rho_i^2 (sum_j m_j GK e_ij) is applied once after the row.
// BETA: some material has a quadratic viscosity term (beta != 0); without
// it Pi = 2 alpha c h vdot / ((r^2 + 0.01 h^2) D)
template <int LANES, bool GC, bool BETA, class Rows, class Rec>
__device__ inline void accel_mx_lane(const Dev &d, int cur, int i, int sub, const Rows &rows, const Rec &rec,
                                     float (&acc)[3]) {
  float ax = 0, ay = 0, az = 0, sx = 0, sy = 0, sz = 0;
  float Li[6];
  own_corr<GC>(d, i, Li);
  const DevMat &M = d.mats[d.mat[i]];
  const float4 xi = d.xhf[cur][i], vi = d.vmf[i];
  const StressRecF ri = d.srecf[i];
  const float h = (float)d.xh[cur][i].w;
  const GkF k = gk_consts(h, d.dim);
  const float h2c = 0.01f * h * h, hh = 2.0f * h;
  const float acs = (float)(M.alpha * M.Cs), bh = 0.5f * (float)M.beta, hha = hh * acs;
  walk_groups<LANES>(rows, d.nnb[i], sub, rows.self(), rows.group(2 * sub), rows.group(2 * sub + 1), [&](const typename Rows::G &c) {
    float4 X[4], V[4], T[4];
    float2 T2[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) rec.load(entry(c, u), X[u], V[u], T[u], T2[u]);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float dx = xi.x - X[u].x, dy = xi.y - X[u].y, dz = xi.z - X[u].z;
      const float r2 = dx * dx + dy * dy + dz * dz;
      const float GK = gk_f(r2, k);
      // Monaghan viscosity for approaching pairs: with D = rho_i + rho_j,
      // mu = h vdot / (r^2 + 0.01 h^2), Pi = mu (alpha c + beta mu) / (D/2)
      const float vdot = (vi.x - V[u].x) * dx + (vi.y - V[u].y) * dy + (vi.z - V[u].z) * dz;
      const float D = ri.rho + X[u].w;
      const float rd = __builtin_amdgcn_rcpf((r2 + h2c) * D);
      float pv;
      if constexpr (BETA) {
        const float hv = (hh * vdot) * rd;
        pv = hv * fmaf(bh, hv * D, acs);
      } else {
        pv = (hha * vdot) * rd;
      }
      const float pi = vdot < 0.0f ? pv : 0.0f;
      const float w = V[u].w * GK;
      float ex, ey, ez;
      corr_dir<GC>(Li, dx, dy, dz, ex, ey, ez);
      const float ux = fmaf(T[u].x, ex, fmaf(T[u].w, ey, fmaf(T2[u].x, ez, pi * ex)));
      const float uy = fmaf(T[u].w, ex, fmaf(T[u].y, ey, fmaf(T2[u].y, ez, pi * ey)));
      const float uz = fmaf(T2[u].x, ex, fmaf(T2[u].y, ey, fmaf(T[u].z, ez, pi * ez)));
      ax = fmaf(w, ux, ax);
      ay = fmaf(w, uy, ay);
      az = fmaf(w, uz, az);
      sx = fmaf(w, ex, sx);
      sy = fmaf(w, ey, sy);
      sz = fmaf(w, ez, sz);
    }
  });
  acc[0] = ax + (ri.t[XX] * sx + ri.t[XY] * sy + ri.t[XZ] * sz);
  acc[1] = ay + (ri.t[XY] * sx + ri.t[YY] * sy + ri.t[YZ] * sz);
  acc[2] = az + (ri.t[XZ] * sx + ri.t[YZ] * sy + ri.t[ZZ] * sz);
}

// FP64: HBM gathers, LANES threads per particle
template <int LANES>
__global__ __launch_bounds__(kBlock *LANES) void k_accel_f64(Dev d, int cur) {
  __shared__ double red[(LANES > 1 ? LANES - 1 : 1) * 3 * kBlock];
  const int t = xcd_tile(blockIdx.x, gridDim.x), sub = threadIdx.x / kBlock;
  const int i = t * kBlock + (int)(threadIdx.x % kBlock);
  double a[3] = {0, 0, 0};
  if (i < d.n) {
    const HbmJ<false> g{d, cur, i};
    if (d.gc_on) {
      if (d.ti_on) accel_lane<false, true, true>(d, cur, i, g, sub, LANES, a);
      else accel_lane<false, false, true>(d, cur, i, g, sub, LANES, a);
    } else {
      if (d.ti_on) accel_lane<false, true, false>(d, cur, i, g, sub, LANES, a);
      else accel_lane<false, false, false>(d, cur, i, g, sub, LANES, a);
    }
  }
  combine_lanes<LANES>(a, red);
  // plane strain: the pair forces have no z part (Source/InteractionAlt.cpp:
  // 184; the corrected-gradient terms keep theirs)
  if (d.dim == 2 && !d.gc_on) a[2] = 0.0;
  if (i < d.n && sub == 0) d.acc[i] = make_double4(a[0], a[1], a[2], 0.0);
}

// FP64, uniform h: 112 bytes of LDS per staged particle, one block per CU.
// The particle's own values and first row words are loaded before the tile
// is staged, so their latency and the staging's overlap.
template <bool GC, bool BETA, bool DAM>
__global__ __launch_bounds__(kBlock *kLanesLds64) void k_accel64(Dev d, int cur) {
  __shared__ double2 rec[kRecAccel * kStageMax];
  __shared__ double dm[DAM ? kStageMax : 1];
  __shared__ double red[(kLanesLds64 - 1) * 3 * kBlock];
  const int t = xcd_tile(blockIdx.x, gridDim.x), sub = threadIdx.x / kBlock;
  const int i = t * kBlock + (int)(threadIdx.x % kBlock);
  const int U = d.stage_cnt[t];
  const bool on = i < d.n && d.group[i] >= 0;
  const int cnt = on ? d.nnb[i] : 0;
  const double4 xi = d.xh[cur][i], vi = d.vm[i];
  const StressRec ri = d.srec[i];
  double a[3] = {0, 0, 0};
  if (U < 0) {
    const HbmRows rows{reinterpret_cast<const int4 *>(d.nbr) + i, d.npad, i};
    if (on)
      accel64_lane<GC, BETA, DAM>(d, i, sub, cnt, xi, vi, ri, rows, rows.group(2 * sub), rows.group(2 * sub + 1),
                                    RecHbm64<PASS_ACCEL>{d, cur}, a);
  } else {
    const LdsRows rows{reinterpret_cast<const ushort4 *>(d.nbrl) + i, d.npad, (int)d.selfl[i]};
    const ushort4 a0 = rows.group(2 * sub), b0 = rows.group(2 * sub + 1);
    stage64<kBlock * kLanesLds64, PASS_ACCEL>(d, cur, t, U, rec, nullptr, dm);
    if (on) accel64_lane<GC, BETA, DAM>(d, i, sub, cnt, xi, vi, ri, rows, a0, b0, RecLds64<PASS_ACCEL>{rec, nullptr, dm}, a);
  }
  combine_lanes<kLanesLds64>(a, red);
  if (d.dim == 2 && !d.gc_on) a[2] = 0.0;  // plane strain, as k_accel_f64
  if (i < d.n && sub == 0) d.acc[i] = make_double4(a[0], a[1], a[2], 0.0);
}

// mixed precision: LDS-staged gathers where the tile is staged, else HBM
template <int LANES, bool GC, bool BETA>
__device__ inline void k_accel_mx_body(const Dev &d, int cur) {
  __shared__ float4 lx[kStageMax + 1], lv[kStageMax + 1], lt[kStageMax + 1];
  __shared__ float2 lt2[kStageMax + 1];
  __shared__ float red[(LANES > 1 ? LANES - 1 : 1) * 3 * kBlock];
  const int t = xcd_tile(blockIdx.x, gridDim.x), sub = threadIdx.x / kBlock;
  const int i = t * kBlock + (int)(threadIdx.x % kBlock);
  const int U = d.stage_cnt[t];
  float a[3] = {0, 0, 0};
  if (U < 0) {
    if (i < d.n && d.group[i] >= 0) {
      const HbmRows rows{reinterpret_cast<const int4 *>(d.nbr) + i, d.npad, i};
      const AccelHbm rec{d.xhf[cur], d.vmf, reinterpret_cast<const float4 *>(d.srecf)};
      accel_mx_lane<LANES, GC, BETA>(d, cur, i, sub, rows, rec, a);
    }
  } else {
    stage_accel<kBlock * LANES>(d, t, U, d.xhf[cur], lx, lv, lt, lt2);
    if (i < d.n && d.group[i] >= 0) {
      const LdsRows rows{reinterpret_cast<const ushort4 *>(d.nbrl) + i, d.npad, (int)d.selfl[i]};
      const AccelLds rec{lx, lv, lt, lt2};
      accel_mx_lane<LANES, GC, BETA>(d, cur, i, sub, rows, rec, a);
    }
  }
  combine_lanes<LANES>(a, red);
  if (d.dim == 2 && !d.gc_on) a[2] = 0.0f;  // plane strain, as the FP64 pass
  if (i < d.n && sub == 0) d.acc[i] = make_double4((double)a[0], (double)a[1], (double)a[2], 0.0);
}

// the kernels with and without the quadratic viscosity term.  The staged
// records fill ~51 KB of LDS, so three blocks share a CU: with two or more
// lanes per particle the kernels are held to the registers of three waves
// per SIMD
template <int LANES, bool GC>
__global__ __launch_bounds__(kBlock *LANES) __attribute__((amdgpu_waves_per_eu(LANES >= 2 ? 3 : 1))) void k_accel_mx_b(
    Dev d, int cur) {
  k_accel_mx_body<LANES, GC, true>(d, cur);
}
template <int LANES, bool GC>
__global__ __launch_bounds__(kBlock *LANES) __attribute__((amdgpu_waves_per_eu(LANES >= 2 ? 3 : 1))) void k_accel_mx_nb(
    Dev d, int cur) {
  k_accel_mx_body<LANES, GC, false>(d, cur);
}

// mixed precision with tensile instability: HBM gathers (the staged
// records do not carry the TI stress)
template <int LANES>
__global__ __launch_bounds__(kBlock *LANES) void k_accel_mx_ti(Dev d, int cur) {
  __shared__ float red[(LANES > 1 ? LANES - 1 : 1) * 3 * kBlock];
  const int t = xcd_tile(blockIdx.x, gridDim.x), sub = threadIdx.x / kBlock;
  const int i = t * kBlock + (int)(threadIdx.x % kBlock);
  float a[3] = {0, 0, 0};
  if (i < d.n) {
    const HbmJ<true> g{d, cur, i};
    if (d.gc_on) accel_lane<true, true, true>(d, cur, i, g, sub, LANES, a);
    else accel_lane<true, true, false>(d, cur, i, g, sub, LANES, a);
  }
  combine_lanes<LANES>(a, red);
  if (d.dim == 2 && !d.gc_on) a[2] = 0.0f;  // plane strain, as the FP64 pass
  if (i < d.n && sub == 0) d.acc[i] = make_double4((double)a[0], (double)a[1], (double)a[2], 0.0);
}

#define WF_LANES_SWITCH(lanes, KERNEL, ...)                                    \
  switch (lanes) {                                                            \
    case 1: KERNEL<1><<<nblk(d.n), kBlock * 1, 0, st>>>(__VA_ARGS__); break;  \
    case 2: KERNEL<2><<<nblk(d.n), kBlock * 2, 0, st>>>(__VA_ARGS__); break;  \
    default: KERNEL<4><<<nblk(d.n), kBlock * 4, 0, st>>>(__VA_ARGS__); break; \
  }
// the FP64 passes from LDS, by gradient correction and the pass's own options
// (compile-time, so that the row walk has no branch)
template <class F>
static void gc_switch(bool gc, F &&f) {
  if (gc) f(std::true_type{});
  else f(std::false_type{});
}
// the mixed-precision passes are also instantiated per gradient correction
#define WF_LANES_GC_SWITCH(lanes, gc, KERNEL, ...)                   \
  if (gc) {                                                         \
    switch (lanes) {                                                \
      case 1: KERNEL<1, true><<<nblk(d.n), kBlock * 1, 0, st>>>(__VA_ARGS__); break;  \
      case 2: KERNEL<2, true><<<nblk(d.n), kBlock * 2, 0, st>>>(__VA_ARGS__); break;  \
      default: KERNEL<4, true><<<nblk(d.n), kBlock * 4, 0, st>>>(__VA_ARGS__); break; \
    }                                                               \
  } else {                                                          \
    switch (lanes) {                                                \
      case 1: KERNEL<1, false><<<nblk(d.n), kBlock * 1, 0, st>>>(__VA_ARGS__); break;  \
      case 2: KERNEL<2, false><<<nblk(d.n), kBlock * 2, 0, st>>>(__VA_ARGS__); break;  \
      default: KERNEL<4, false><<<nblk(d.n), kBlock * 4, 0, st>>>(__VA_ARGS__); break; \
    }                                                               \
  }

// StartAcceleration's tensile-instability stress, 3D branch
// (Source/Domain.cpp:1529-1563): principal stresses s_k > 0 become
// -TI s_k / rho^2, the others 0, rotated back with the eigenvectors
// ((Vec Val) Vec^T).  The eigen-decomposition is cyclic Jacobi (Golub & Van
// Loan, Alg. 8.5.3) in FP64; the result is a spectral function of sigma, so
// it does not depend on the eigenvectors' signs or order.
WF_KERNEL void k_tir(Dev d, int cur) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= d.n) return;
  const long long np = d.npad;
  double out[6] = {0, 0, 0, 0, 0, 0};
  if (d.group[i] >= 0 && d.mats[d.mat[i]].ti > 0.0) {
    const StressRec r = d.srec[i];
    double A[3][3] = {{r.s[XX], r.s[XY], r.s[XZ]}, {r.s[XY], r.s[YY], r.s[YZ]}, {r.s[XZ], r.s[YZ], r.s[ZZ]}};
    double V[3][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}};
    for (int sweep = 0; sweep < 64; ++sweep) {
      const double off = A[0][1] * A[0][1] + A[0][2] * A[0][2] + A[1][2] * A[1][2];
      const double dia = A[0][0] * A[0][0] + A[1][1] * A[1][1] + A[2][2] * A[2][2];
      if (off == 0.0 || off <= 1e-40 * dia) break;
      for (int p = 0; p < 2; ++p)
        for (int q = p + 1; q < 3; ++q) {
          if (A[p][q] == 0.0) continue;
          const double th = (A[q][q] - A[p][p]) / (2.0 * A[p][q]);
          const double t = (th >= 0 ? 1.0 : -1.0) / (fabs(th) + sqrt(th * th + 1.0));
          const double c = 1.0 / sqrt(t * t + 1.0), s = t * c;
          for (int k = 0; k < 3; ++k) {
            const double akp = A[k][p], akq = A[k][q];
            A[k][p] = c * akp - s * akq;
            A[k][q] = s * akp + c * akq;
          }
          for (int k = 0; k < 3; ++k) {
            const double apk = A[p][k], aqk = A[q][k];
            A[p][k] = c * apk - s * aqk;
            A[q][k] = s * apk + c * aqk;
          }
          A[p][q] = A[q][p] = 0.0;
          for (int k = 0; k < 3; ++k) {
            const double vkp = V[k][p], vkq = V[k][q];
            V[k][p] = c * vkp - s * vkq;
            V[k][q] = s * vkp + c * vkq;
          }
        }
    }
    const double pc = d.mats[d.mat[i]].ti / (r.rho * r.rho);
    double w[3];
    for (int k = 0; k < 3; ++k) w[k] = A[k][k] > 0 ? -pc * A[k][k] : 0.0;
    const int ia[6] = {0, 1, 2, 0, 0, 1}, ib[6] = {0, 1, 2, 1, 2, 2};
    for (int m = 0; m < 6; ++m) {
      double s = 0.0;
      for (int k = 0; k < 3; ++k) s += (V[ia[m]][k] * w[k]) * V[ib[m]][k];
      out[m] = s;
    }
  }
  for (int m = 0; m < 6; ++m) d.tir[(long long)m * np + i] = out[m];
  if (d.mixed)
    for (int m = 0; m < 6; ++m) d.tirf[(long long)m * np + i] = (float)out[m];
}

void launch_tir(const Dev &d, hipStream_t st, int cur) { k_tir<<<nblk(d.n), kBlock, 0, st>>>(d, cur); }

void launch_accel(const Dev &d, hipStream_t st, int cur) {
  if (d.mixed && d.ti_on) {
    WF_LANES_SWITCH(d.lanes_mx, k_accel_mx_ti, d, cur)
  } else if (d.mixed && d.beta_on) {
    WF_LANES_GC_SWITCH(d.lanes_mx, d.gc_on, k_accel_mx_b, d, cur)
  } else if (d.mixed) {
    WF_LANES_GC_SWITCH(d.lanes_mx, d.gc_on, k_accel_mx_nb, d, cur)
  } else if (d.lds64 && !d.ti_on) {
    gc_switch(d.gc_on, [&](auto gc) {
      constexpr bool GC = decltype(gc)::value;
      const dim3 g(nblk(d.n)), b(kBlock * kLanesLds64);
      if (d.damage) {
        if (d.beta_on) k_accel64<GC, true, true><<<g, b, 0, st>>>(d, cur);
        else k_accel64<GC, false, true><<<g, b, 0, st>>>(d, cur);
      } else {
        if (d.beta_on) k_accel64<GC, true, false><<<g, b, 0, st>>>(d, cur);
        else k_accel64<GC, false, false><<<g, b, 0, st>>>(d, cur);
      }
    });
  } else {
    // FP64 with the tensile-instability stress or smoothing lengths that
    // differ within a material
    WF_LANES_SWITCH(d.lanes_f64, k_accel_f64, d, cur)
  }
}

// ---------------------------------------------------------------------------
// velocity kicks with the UserAcc BC semantics (Source/WeldForm.cpp:51-92)
// and the reaction observer at the first GeneralAfter of the step.
//   Leapfrog  (Source/SolverLeapfrog.cpp:228-273):
//       [first step] v -= a*0.5*dt ;  v += a*0.5*(dt_prev + dt)
//   KickDrift (Source/SolverKickDrift.cpp:208-231): v += a*0.5*dt_prev


WF_KERNEL void k_kick(Dev d, BcTable bc, int scheme, double dt_prev, double dt, int kphase) {
  __shared__ double sh[kBlock / 64];
  __shared__ double bcv[kMaxBc][3];
  __shared__ int bcon[kMaxBc];
  const bool observe = kphase == K_WHOLE || kphase == K_FIRST || kphase == K_OBSERVE;
  const int phase = kphase == K_WHOLE_NOOBS ? K_WHOLE : (kphase == K_FIRST_NOOBS ? K_FIRST : kphase);
  const int isfirst = d.flags->step == 0;
  if (dt < 0) {
    dt = d.flags->dt;
    dt_prev = d.flags->dt_prev;
  }
  if (threadIdx.x < bc.n) {
    // velocity of each BC at the step's time (UserAcc, Source/WeldForm.cpp:67-82)
    const int b = threadIdx.x;
    int on = 1;
    double f = 1.0;
    if (bc.type[b] == 0 && bc.value_type[b] == 1) {
      if (bc.amp[b] < 0) on = 0;
      else f = bc.amp_factor[b] * amp_value(d.amps[bc.amp[b]], d.flags->time);
    }
    for (int k = 0; k < 3; ++k) bcv[b][k] = bc.value_type[b] == 1 ? f * bc.v[b][k] : bc.v[b][k];
    bcon[b] = on;
  }
  __syncthreads();
  const int i = blockIdx.x * kBlock + threadIdx.x;
  double4 a = make_double4(0, 0, 0, 0);
  double m = 0.0;
  int id = -0x7fffffff;
  if (i < d.n) {
    a = d.acc[i];
    const double4 vm = d.vm[i];
    m = vm.w;
    id = d.id[i];
  }
  if (i < d.n && phase != K_OBSERVE) {
    const double4 vm = d.vm[i];
    double v[3] = {vm.x, vm.y, vm.z};
    double av[3] = {a.x, a.y, a.z};
    if (!isfinite(a.x) || !isfinite(a.y) || !isfinite(a.z)) d.flags->nan = 1;
    bool fixed = false;
    for (int b = 0; b < bc.n; ++b) {
      if (bc.zone[b] != id || !bcon[b]) continue;
      if (bc.type[b] == 0) {
        fixed = true;
        for (int k = 0; k < 3; ++k) {
          av[k] = 0.0;
          v[k] = bcv[b][k];
        }
      } else if (bc.type[b] == 2) {
        d.T[i] = bc.T[b];
      }
    }
    if (!fixed) {
      if (scheme == WF_LEAPFROG) {
        if (isfirst && phase != K_SECOND)
          for (int k = 0; k < 3; ++k) v[k] -= av[k] * 0.5 * dt;
        if (phase != K_FIRST)
          for (int k = 0; k < 3; ++k) v[k] += av[k] * 0.5 * (dt_prev + dt);
      } else if (phase != K_FIRST) {
        for (int k = 0; k < 3; ++k) v[k] += av[k] * 0.5 * dt_prev;
      }
    }
    d.vm[i] = make_double4(v[0], v[1], v[2], vm.w);
    if (d.mixed) d.vmf[i] = make_float4((float)v[0], (float)v[1], (float)v[2], (float)vm.w);
    d.acc[i] = make_double4(av[0], av[1], av[2], 0.0);
  }
  for (int z = 0; z < bc.nz && observe; ++z) {
    const bool in = (id == bc.rzone[z]);
    const double fx = block_reduce<0>(in ? m * a.x : 0.0, sh);
    const double fy = block_reduce<0>(in ? m * a.y : 0.0, sh);
    const double fz = block_reduce<0>(in ? m * a.z : 0.0, sh);
    if (threadIdx.x == 0) {
      part(d, P_REACT + 3 * z, blockIdx.x) = fx;
      part(d, P_REACT + 3 * z + 1, blockIdx.x) = fy;
      part(d, P_REACT + 3 * z + 2, blockIdx.x) = fz;
    }
  }
}

// KickDrift's second half kick, v += a*dt/2 (Source/SolverKickDrift.cpp:261-265)
WF_KERNEL void k_kick2(Dev d, double dt) {
  if (dt < 0) dt = d.flags->dt;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= d.n) return;
  const double4 a = d.acc[i];
  double4 v = d.vm[i];
  v.x += a.x * dt / 2.;
  v.y += a.y * dt / 2.;
  v.z += a.z * dt / 2.;
  d.vm[i] = v;
  if (d.mixed) d.vmf[i] = make_float4((float)v.x, (float)v.y, (float)v.z, (float)v.w);
}

void launch_kick(const Dev &d, hipStream_t st, const BcTable &bc, int scheme, double dt_prev, double dt, int phase) {
  k_kick<<<d.nblocks, kBlock, 0, st>>>(d, bc, scheme, dt_prev, dt, phase);
}

// CheckMinTSVel / CheckMinTSAccel (Source/Domain.cpp:265-319): per particle
// the smallest neighbour distance over CFL (Cs + |v|), or sqrt_h_a
// sqrt(h / |a|) (the acceleration criterion, evaluated last, wins when both
// are on); block minima, then AdaptiveTimeStep (:206-239) in one thread.
//
// The distance pass reads FP64 positions from the tile's LDS copy, four lanes
// per particle (tiles that are not staged: from HBM).  The square root is
// monotonic, so the least square gives the least distance exactly.  One lane
// per particle gathering the positions from HBM, a root per neighbour, took
// 35 us at 35k particles, now 7.2 us.
struct PosLds {
  const double2 *xy;
  const double *z;
  __device__ double3 load(int p) const { return make_double3(xy[p].x, xy[p].y, z[p]); }
};
struct PosHbm {
  const double4 *x;
  __device__ double3 load(int j) const {
    const double4 a = x[j];
    return make_double3(a.x, a.y, a.z);
  }
};
template <class Rows, class Rec>
__device__ inline double least_r2(const Rows &rows, const Rec &rec, int own, int cnt, int sub, const double4 &xi,
                                  typename Rows::G a0, typename Rows::G b0) {
#pragma clang fp contract(off)
  double mn = INFINITY;
  walk_groups<kLanesLds64>(rows, cnt, sub, rows.self(), a0, b0, [&](const typename Rows::G &c) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int p = entry(c, u);
      const double3 x = rec.load(p);
      const double dx = x.x - xi.x, dy = x.y - xi.y, dz = x.z - xi.z;
      const double r2 = dx * dx + dy * dy + dz * dz;
      mn = fmin(mn, p == own ? INFINITY : r2);  // (padding entries are the particle itself)
    }
  });
  return mn;
}
__global__ __launch_bounds__(kBlock *kLanesLds64) void k_ts_vel(Dev d, int cur) {
#pragma clang fp contract(off)
  constexpr int NT = kBlock * kLanesLds64;
  __shared__ double2 xy[kStageMax];
  __shared__ double z[kStageMax];
  __shared__ double red[(kLanesLds64 - 1) * kBlock];
  __shared__ double sh[NT / 64];
  const int t = xcd_tile(blockIdx.x, gridDim.x), sub = threadIdx.x / kBlock, lane = threadIdx.x % kBlock;
  const int i = t * kBlock + lane;
  const int U = d.stage_cnt[t];
  const int cnt = i < d.n ? d.nnb[i] : 0;
  const double4 xi = d.xh[cur][i];
  double mn;
  if (U < 0) {
    const HbmRows rows{reinterpret_cast<const int4 *>(d.nbr) + i, d.npad, i};
    mn = least_r2(rows, PosHbm{d.xh[cur]}, i, cnt, sub, xi, rows.group(2 * sub), rows.group(2 * sub + 1));
  } else {
    const LdsRows rows{reinterpret_cast<const ushort4 *>(d.nbrl) + i, d.npad, (int)d.selfl[i]};
    const ushort4 a0 = rows.group(2 * sub), b0 = rows.group(2 * sub + 1);
    stage_set<NT>(d.stage, t, U, [&](int p, int j) {
      const double4 x = d.xh[cur][j];
      xy[p] = make_double2(x.x, x.y);
      z[p] = x.z;
    });
    mn = least_r2(rows, PosLds{xy, z}, rows.own, cnt, sub, xi, a0, b0);
  }
  if (sub > 0) red[(sub - 1) * kBlock + lane] = mn;
  __syncthreads();
  double test = INFINITY;
  if (sub == 0 && i < d.n) {
    for (int q = 0; q < kLanesLds64 - 1; ++q) mn = fmin(mn, red[q * kBlock + lane]);
    const double4 v = d.vm[i];
    test = d.cfl * fmin(1000., sqrt(mn)) / (d.mats[d.mat[i]].Cs + sqrt(v.x * v.x + v.y * v.y + v.z * v.z));
  }
  const double r = block_reduce<2>(test, sh);
  if (threadIdx.x == 0) part(d, P_DTMIN, t) = r;
}
WF_KERNEL void k_ts_acc(Dev d, int cur) {
#pragma clang fp contract(off)
  __shared__ double sh[kBlock / 64];
  const int i = blockIdx.x * kBlock + threadIdx.x;
  double test = INFINITY;
  if (i < d.n) {
    const double4 a = d.acc[i];
    test = d.sqrt_h_a * sqrt(d.xh[cur][i].w / sqrt(a.x * a.x + a.y * a.y + a.z * a.z));
  }
  const double r = block_reduce<2>(test, sh);
  if (threadIdx.x == 0) part(d, P_DTMIN, blockIdx.x) = r;
}

__global__ __launch_bounds__(1024) void k_ts_adapt(Dev d) {
  __shared__ double sh[16];
  double v = INFINITY;
  for (int b = threadIdx.x; b < d.nblocks; b += blockDim.x) v = fmin(v, part(d, P_DTMIN, b));
  const double r = block_reduce<2>(v, sh);
  // the contact criterion: the least dt_fext of this step's pairs
  const bool cont_ts = d.contact && (d.auto_ts & 4);
  double fts = INFINITY;
  if (cont_ts) {
    for (int b = threadIdx.x; b < d.nblocks; b += blockDim.x) fts = fmin(fts, part(d, P_FTS, b));
    fts = block_reduce<2>(fts, sh);
  }
  if (threadIdx.x != 0) return;
  DevFlags *f = d.flags;
  if (fts < INFINITY) f->min_force_ts = fts;
  const double dint = f->dtint, dmin = fmin(dint, r);
  double dt = f->dt;
  f->dt_prev = dt;
  if (dint > dmin) {
    if (dt < dmin) dt = 2.0 * dt * dmin / (dt + dmin);
    else dt = dmin;
  } else {
    if (dint != dt) dt = 2.0 * dt * dint / (dt + dint);
    else dt = dint;
  }
  if (cont_ts && f->min_force_ts < dt) dt = f->min_force_ts;
  if (dt < d.min_ts) dt = d.min_ts;
  f->dt = dt;
}

void launch_time_step(const Dev &d, hipStream_t st, int cur) {
  if (d.auto_ts & 2) k_ts_acc<<<d.nblocks, kBlock, 0, st>>>(d, cur);
  else k_ts_vel<<<d.nblocks, kBlock * kLanesLds64, 0, st>>>(d, cur);
  k_ts_adapt<<<1, 1024, 0, st>>>(d);
}

void launch_kick2(const Dev &d, hipStream_t st, double dt) { k_kick2<<<nblk(d.n), kBlock, 0, st>>>(d, dt); }

// ---------------------------------------------------------------------------
// pass 2: density rate + density update + drift
// (CalcDensInc + DensReduction, Source/InteractionAlt.cpp:483-640;
//  Source/SolverLeapfrog.cpp:280-301).  Reads x_n, v_{n+1/2}, m/rho_n and
// writes rho_{n+1}, m/rho_{n+1}, x_{n+1} into the other buffer.

template <bool GC, class G>
__device__ inline double dens_lane(const Dev &d, int cur, int i, const G &g, int sub, int lanes) {
  using S = Src<false>;
  double s = 0;
  if (d.group[i] >= 0) {
    double Li[6];
    own_corr<GC>(d, i, Li);
    const double4 xi = S::x(d, cur, i), vi = S::v(d, i);
    const KH<double> ki = kern_h_t<double>(xi.w, d.dim);
    for_each_nb(g, d.nnb[i], sub, lanes, [&](int j) {
      const double4 xj = g.x(j), vj = g.v(j);
      const double volj = g.vol(j);
      const double dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
      const double GK = gk_t<double>(dx * dx + dy * dy + dz * dz, S::kh(ki, xi, xj));
      double ex, ey, ez;
      corr_dir<GC>(Li, dx, dy, dz, ex, ey, ez);
      const double t = (vi.x - vj.x) * (GK * ex) + (vi.y - vj.y) * (GK * ey) + (vi.z - vj.z) * (GK * ez);
      double wv = volj;
      // damage weight of the pair (Source/InteractionAlt.cpp:558-572)
      if (d.damage) {
        const double df = dam_weight(d.damD[i], g.dam(j));
        wv = df > 0.0 ? df * volj : 0.0;
      }
      s += wv * t;
    });
  }
  return s;
}

// the particle's own FP64 state the update reads
struct DensOwn {
  double rho;
  double4 x, v, u;
};
__device__ inline DensOwn dens_own(const Dev &d, int cur, int i) {
  return DensOwn{d.rho[cur][i], d.xh[cur][i], d.vm[i], d.disp[i]};
}

template <bool MX>
__device__ inline void dens_update(const Dev &d, int cur, int i, double s, double dt, int do_update,
                                   const DensOwn &o) {
  if (dt < 0) dt = d.flags->dt;
  const double rhoi = o.rho;
  const double drho = s * rhoi;
  d.drho[i] = drho;
  if (!do_update) return;
  const int nxt = cur ^ 1;
  const double4 xd = o.x;
  const double4 vd = o.v;
  const double rn = rhoi + dt * drho;
  const double vn = vd.w / rn;
  d.rho[nxt][i] = rn;
  d.vol[nxt][i] = vn;
  const double ux = vd.x * dt, uy = vd.y * dt, uz = vd.z * dt;
  double4 u = o.u;
  u.x += ux;
  u.y += uy;
  u.z += uz;
  d.disp[i] = u;
  const double4 xn = make_double4(xd.x + ux, xd.y + uy, xd.z + uz, xd.w);
  d.xh[nxt][i] = xn;
  if (MX) {
    const double *o = d.mats[d.mat[i]].xc;
    d.xhf[nxt][i] = make_float4((float)(xn.x - o[0]), (float)(xn.y - o[1]), (float)(xn.z - o[2]), (float)vn);
    const DevMat &M = d.mats[d.mat[i]];
    d.prf[i] = (float)((M.P0 + M.Cs * M.Cs * (rn - M.ref_density)) / (rn * rn));
  }
}

template <int LANES>
__global__ __launch_bounds__(kBlock *LANES) void k_dens_f64(Dev d, int cur, double dt, int do_update) {
  __shared__ double red[(LANES > 1 ? LANES - 1 : 1) * kBlock];
  const int t = xcd_tile(blockIdx.x, gridDim.x), sub = threadIdx.x / kBlock;
  const int i = t * kBlock + (int)(threadIdx.x % kBlock);
  double s[1] = {0};
  if (i < d.n) {
    const HbmJ<false> g{d, cur, i};
    s[0] = d.gc_on ? dens_lane<true>(d, cur, i, g, sub, LANES) : dens_lane<false>(d, cur, i, g, sub, LANES);
  }
  combine_lanes<LANES>(s, red);
  if (i < d.n && sub == 0) dens_update<false>(d, cur, i, s[0], dt, do_update, dens_own(d, cur, i));
}

// FP64, uniform h: 56 bytes of LDS per staged particle, three blocks per CU
// (two with damage)
template <bool GC, bool DAM>
__global__ __launch_bounds__(kBlock *kLanesLds64) void k_dens64(Dev d, int cur, double dt, int do_update) {
  __shared__ double2 rec[kRecDens * kStageMax];
  __shared__ double sc[kStageMax];
  __shared__ double dm[DAM ? kStageMax : 1];
  __shared__ double red[(kLanesLds64 - 1) * kBlock];
  const int t = xcd_tile(blockIdx.x, gridDim.x), sub = threadIdx.x / kBlock;
  const int i = t * kBlock + (int)(threadIdx.x % kBlock);
  const int U = d.stage_cnt[t];
  const bool on = i < d.n && d.group[i] >= 0;
  const int cnt = on ? d.nnb[i] : 0;
  const double4 xi = d.xh[cur][i], vi = d.vm[i];
  double s[1] = {0};
  if (U < 0) {
    const HbmRows rows{reinterpret_cast<const int4 *>(d.nbr) + i, d.npad, i};
    if (on)
      s[0] = dens64_lane<GC, DAM>(d, i, sub, cnt, xi, vi, rows, rows.group(2 * sub), rows.group(2 * sub + 1),
                                    RecHbm64<PASS_DENS>{d, cur});
  } else {
    const LdsRows rows{reinterpret_cast<const ushort4 *>(d.nbrl) + i, d.npad, (int)d.selfl[i]};
    const ushort4 a0 = rows.group(2 * sub), b0 = rows.group(2 * sub + 1);
    stage64<kBlock * kLanesLds64, PASS_DENS>(d, cur, t, U, rec, sc, dm);
    if (on) s[0] = dens64_lane<GC, DAM>(d, i, sub, cnt, xi, vi, rows, a0, b0, RecLds64<PASS_DENS>{rec, sc, dm});
  }
  combine_lanes<kLanesLds64>(s, red);
  if (i < d.n && sub == 0) dens_update<false>(d, cur, i, s[0], dt, do_update, DensOwn{d.rho[cur][i], xi, vi, d.disp[i]});
}

// records of the density and rate passes: X = (x, y, z, m/rho), V = (v, m)
// and, for the rates, P / rho^2
struct XvLds {
  const float4 *lx, *lv;
  const float *lp;
  __device__ void load(int l, float4 &X, float4 &V) const {
    X = lx[l];
    V = lv[l];
  }
  __device__ float pr(int l) const { return lp[l]; }
};
struct XvHbm {
  const float4 *gx, *gv;
  const float *gp;
  __device__ void load(int j, float4 &X, float4 &V) const {
    X = gx[j];
    V = gv[j];
  }
  __device__ float pr(int j) const { return gp[j]; }
};

// CalcDensInc + DensReduction in FP32 (Source/InteractionAlt.cpp:483-640):
// sum_j (m_j / rho_j) v_ij . (GK e_ij); the caller multiplies by rho_i
template <int LANES, bool GC, class Rows, class Rec>
__device__ inline float dens_mx_lane(const Dev &d, int cur, int i, int sub, const Rows &rows, const Rec &rec) {
  float s = 0;
  float Li[6];
  own_corr<GC>(d, i, Li);
  const float4 xi = d.xhf[cur][i], vi = d.vmf[i];
  const GkF k = gk_consts((float)d.xh[cur][i].w, d.dim);
  walk_groups<LANES>(rows, d.nnb[i], sub, rows.self(), rows.group(2 * sub), rows.group(2 * sub + 1), [&](const typename Rows::G &c) {
    float4 X[4], V[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) rec.load(entry(c, u), X[u], V[u]);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float dx = xi.x - X[u].x, dy = xi.y - X[u].y, dz = xi.z - X[u].z;
      const float GK = gk_f(dx * dx + dy * dy + dz * dz, k);
      float ex, ey, ez;
      corr_dir<GC>(Li, dx, dy, dz, ex, ey, ez);
      const float t = (vi.x - V[u].x) * ex + (vi.y - V[u].y) * ey + (vi.z - V[u].z) * ez;
      s = fmaf(X[u].w * GK, t, s);
    }
  });
  return s;
}

template <int LANES, bool GC>
__global__ __launch_bounds__(kBlock *LANES) void k_dens_mx(Dev d, int cur, double dt, int do_update) {
  __shared__ float4 lx[kStageMax + 1], lv[kStageMax + 1];
  __shared__ float red[(LANES > 1 ? LANES - 1 : 1) * kBlock];
  const int t = xcd_tile(blockIdx.x, gridDim.x), sub = threadIdx.x / kBlock;
  const int i = t * kBlock + (int)(threadIdx.x % kBlock);
  const int U = d.stage_cnt[t];
  // the update's FP64 inputs are loaded now and arrive during the row walk
  DensOwn own{};
  if (i < d.n && sub == 0) own = dens_own(d, cur, i);
  float s[1] = {0};
  if (U < 0) {
    if (i < d.n && d.group[i] >= 0) {
      const HbmRows rows{reinterpret_cast<const int4 *>(d.nbr) + i, d.npad, i};
      s[0] = dens_mx_lane<LANES, GC>(d, cur, i, sub, rows, XvHbm{d.xhf[cur], d.vmf, nullptr});
    }
  } else {
    stage_xv<kBlock * LANES>(d, t, U, d.xhf[cur], lx, lv, nullptr);
    if (i < d.n && d.group[i] >= 0) {
      const LdsRows rows{reinterpret_cast<const ushort4 *>(d.nbrl) + i, d.npad, (int)d.selfl[i]};
      s[0] = dens_mx_lane<LANES, GC>(d, cur, i, sub, rows, XvLds{lx, lv, nullptr});
    }
  }
  combine_lanes<LANES>(s, red);
  if (i < d.n && sub == 0) dens_update<true>(d, cur, i, (double)s[0], dt, do_update, own);
}

void launch_dens_drift(const Dev &d, hipStream_t st, int cur, double dt, int do_update) {
  if (d.mixed) {
    WF_LANES_GC_SWITCH(d.lanes_mx, d.gc_on, k_dens_mx, d, cur, dt, do_update)
  } else {
    if (d.lds64) {
      gc_switch(d.gc_on, [&](auto gc) {
        constexpr bool GC = decltype(gc)::value;
        const dim3 g(nblk(d.n)), b(kBlock * kLanesLds64);
        if (d.damage) k_dens64<GC, true><<<g, b, 0, st>>>(d, cur, dt, do_update);
        else k_dens64<GC, false><<<g, b, 0, st>>>(d, cur, dt, do_update);
      });
    } else {
      WF_LANES_SWITCH(d.lanes_f64, k_dens_f64, d, cur, dt, do_update)
    }
  }
}

// ---------------------------------------------------------------------------
// pass 3: strain-rate / rotation-rate gather (CalcRateTensors +
// RateTensorsReduction, Source/InteractionAlt.cpp:263-479) with the kinetic
// energy pair term (Source/Domain.cpp:1752-1808), then the per-particle
// stress update (Particle::CalcStressStrain, Source/Particle.cpp:960-1067)
// with plastic work heat (Source/Particle.cpp:922-939), the temperature
// update of ThermalCalcs (Source/Thermal.cpp:726-734) and the internal
// energy term (Source/Domain.cpp:1810-1829).  The update is a kernel of its
// own, or runs at the end of the gather kernel (see launch_rates).

// one particle's rate-tensor gather: v[0..5] strain rate, v[6..8] rotation
// rate (w01, w02, w12), v[9] the kinetic-energy pair sum
// LK: the Locking sums' weight, m_j / rho_j rounded to float
template <bool GC, bool LK, class G>
__device__ inline void rates_lane(const Dev &d, int buf, int i, const G &g, int sub, int lanes, double (&v)[10]) {
  using Sr = Src<false>;
  double sr[6] = {0, 0, 0, 0, 0, 0}, w[3] = {0, 0, 0};
  double ekin = 0;
  if (d.group[i] >= 0) {
    double Li[6];
    own_corr<GC>(d, i, Li);
    const DevMat &M = d.mats[d.mat[i]];
    const double4 xi = Sr::x(d, buf, i), vi = Sr::v(d, i);
    const double P0 = M.P0, cs2 = M.Cs * M.Cs, rho0 = M.ref_density;
    const double pri = g.pr(g.self(), P0, cs2, rho0);
    const double mi = vi.w;
    const KH<double> ki = kern_h_t<double>(xi.w, d.dim);
    for_each_nb(g, d.nnb[i], sub, lanes, [&](int j) {
      const double4 xj = g.x(j), vj = g.v(j);
      double volj = g.vol(j);
      if constexpr (LK) volj = (double)(float)volj;
      const double dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
      const double GK = gk_t<double>(dx * dx + dy * dy + dz * dz, Sr::kh(ki, xi, xj));
      const double vx = vi.x - vj.x, vy = vi.y - vj.y, vz = vi.z - vj.z;
      const double c = volj * (-0.5 * GK);
      double ex, ey, ez;
      corr_dir<GC>(Li, dx, dy, dz, ex, ey, ez);
      sr[XX] += c * (2.0 * vx * ex);
      sr[YY] += c * (2.0 * vy * ey);
      sr[ZZ] += c * (2.0 * vz * ez);
      sr[XY] += c * (vx * ey + vy * ex);
      sr[XZ] += c * (vx * ez + vz * ex);
      sr[YZ] += c * (vy * ez + vz * ey);
      w[0] += c * (vx * ey - vy * ex);
      w[1] += c * (vx * ez - vz * ex);
      w[2] += c * (vy * ez - vz * ey);
      // kinetic-energy pair term (Source/Domain.cpp:1776-1792): the pair
      // is oriented lower-index first; its sum over particles vanishes
      const double prj = g.pr(j, P0, cs2, rho0);
      const bool lo = g.lower(j);
      const double msec = lo ? vj.w : mi;
      const double term = 0.5 * msec * (pri + prj) * (vx * (GK * dx) + vy * (GK * dy) + vz * (GK * dz));
      ekin += lo ? term : -term;
    });
  }
  for (int k = 0; k < 6; ++k) v[k] = sr[k];
  for (int k = 0; k < 3; ++k) v[6 + k] = w[k];
  v[9] = ekin;
}

template <typename R>
__device__ inline void rates_store(const Dev &d, int i, const R (&v)[10]) {
  const long long np = d.npad;
  for (int k = 0; k < 6; ++k) d.sr[k * np + i] = (double)v[k];
  for (int k = 0; k < 3; ++k) d.rr[k * np + i] = (double)v[6 + k];
}

// Particle::CalcStressStrain and the per-particle terms after it for a free
// particle with strain rate SR and rotation rate W
struct StressSums {
  double e_int = 0.0, e_plw = 0.0, tmax = -INFINITY, tmin = INFINITY;
};
// the state the update reads: the deviatoric stress (t), Sy, pl, T, rho and
// m/rho, or in t the strain alone
struct StressOwn {
  double t[6], sigy, pl, T, rho, vol;
};
__device__ inline StressOwn stress_own(const Dev &d, int buf, int i) {
  StressOwn o;
  for (int k = 0; k < 6; ++k) o.t[k] = d.S[k * d.npad + i];
  o.sigy = d.sigy[i];
  o.pl = d.pl[i];
  o.T = d.T[i];
  o.rho = d.rho[buf][i];
  o.vol = d.vol[buf][i];
  return o;
}
__device__ inline void strain_update(const Dev &d, int i, double dt, const double (&SR)[6], const double (&strain)[6]) {
  for (int k = 0; k < 6; ++k) d.strain[k * d.npad + i] = strain[k] + dt * SR[k];
}
template <bool MX>
__device__ inline void stress_update(const Dev &d, int i, double dt, const double (&SR)[6], const double (&W)[3],
                                     const StressOwn &o, StressSums &e) {
  const long long np = d.npad;
  const DevMat &M = d.mats[d.mat[i]];
  const double rho = o.rho;
  const double P = M.P0 + (M.Cs * M.Cs) * (rho - M.ref_density);
  const double (&S)[6] = o.t;
  // Jaumann terms S*W^T + W*S with W antisymmetric
  const double Sf[3][3] = {{S[XX], S[XY], S[XZ]}, {S[XY], S[YY], S[YZ]}, {S[XZ], S[YZ], S[ZZ]}};
  const double Wf[3][3] = {{0.0, W[0], W[1]}, {-W[0], 0.0, W[2]}, {-W[1], -W[2], 0.0}};
  const int ia[6] = {0, 1, 2, 0, 0, 1}, ib[6] = {0, 1, 2, 1, 2, 2};
  const double c3 = 1.0 / 3.0 * (SR[XX] + SR[YY] + SR[ZZ]);
  const double G2 = 2.0 * M.G;
  double Sn[6];
  for (int k = 0; k < 6; ++k) {
    const int a = ia[k], b = ib[k];
    double jt = 0.0;
    for (int q = 0; q < 3; ++q) jt += Sf[a][q] * Wf[b][q] + Wf[a][q] * Sf[q][b];
    const double dev = k < 3 ? SR[k] - c3 : SR[k];
    Sn[k] = dt * (G2 * dev + jt) + S[k];
  }
  const double effsr = sqrt(0.5 * ((SR[XX] - SR[YY]) * (SR[XX] - SR[YY]) + (SR[YY] - SR[ZZ]) * (SR[YY] - SR[ZZ]) +
                                   (SR[ZZ] - SR[XX]) * (SR[ZZ] - SR[XX])) +
                            3.0 * (SR[XY] * SR[XY] + SR[YZ] * SR[YZ] + SR[XZ] * SR[XZ]));
  const double J2 = 0.5 * (Sn[XX] * Sn[XX] + 2.0 * Sn[XY] * Sn[XY] + 2.0 * Sn[XZ] * Sn[XZ] + Sn[YY] * Sn[YY] +
                           2.0 * Sn[YZ] * Sn[YZ] + Sn[ZZ] * Sn[ZZ]);
  const double sig_trial = sqrt(3.0 * J2);
  double Sy = o.sigy;
  double pl = o.pl;
  const double ratio = Sy / sig_trial;
  const double fac = (1.0 < ratio) ? 1.0 : ratio;
  for (int k = 0; k < 6; ++k) Sn[k] *= fac;
  const double T = o.T;
  if (M.model == WF_HOLLOMON) Sy = hol_yield(M, pl);
  else if (M.model == WF_JOHNSON_COOK) Sy = jc_yield(M, pl, effsr, T);
  double dep = 0.0;
  if (sig_trial > Sy) {
    dep = (sig_trial - Sy) / (3. * M.G + M.Ep);
    pl += dep;
    d.dpl[i] = dep;
    if (M.model == WF_BILINEAR) Sy += dep * M.Ep;
  }
  double sig[6];
  for (int k = 0; k < 6; ++k) sig[k] = k < 3 ? -P + Sn[k] : Sn[k];
  if (dep > 0.0) {
    const double f = dep / Sy;
    const double inc[6] = {f * (sig[XX] - 0.5 * (sig[YY] + sig[ZZ])), f * (sig[YY] - 0.5 * (sig[XX] + sig[ZZ])),
                           f * (sig[ZZ] - 0.5 * (sig[XX] + sig[YY])), 1.5 * f * sig[XY],
                           1.5 * f * sig[XZ],                          1.5 * f * sig[YZ]};
    for (int k = 0; k < 6; ++k) {
      d.eplinc[k * np + i] = inc[k];
      d.epl[k * np + i] += inc[k];
    }
  }
  for (int k = 0; k < 6; ++k) d.S[k * np + i] = Sn[k];
  d.effsr[i] = effsr;
  d.sigy[i] = Sy;
  d.pl[i] = pl;
  d.pres[i] = P;
  // Domain::CalcDamage, Johnson-Cook criterion (Source/Damage.cpp:9-46),
  // after the stress update: the (never reset) delta_pl_strain over the
  // fracture strain at the plastic rate, the triaxiality -P / Sigma_eq
  // (Particle::CalculateEquivalentStress, Source/Particle.cpp:623-633)
  // and T (0 without the thermal solver: the reference's is an
  // uninitialised private copy of a local set to 0)
  if (d.damage && M.dam_model == 1) {
    const double dpl = d.dpl[i];
    if (dpl > 0.0) {
      const double J2e = 0.5 * (Sn[XX] * Sn[XX] + 2.0 * Sn[XY] * Sn[XY] + 2.0 * Sn[XZ] * Sn[XZ] + Sn[YY] * Sn[YY] +
                                2.0 * Sn[YZ] * Sn[YZ] + Sn[ZZ] * Sn[ZZ]);
      const double seq = sqrt(3.0 * J2e);
      if (seq > 1.0e-3) {
        const double ef = jc_fracture_strain(M, dpl / dt, -P / seq, d.thermal ? T : 0.0);
        double D = d.damD[i] + dpl / ef;
        if (D > 1.0) D = 1.0;
        d.damD[i] = D;
      }
    }
  }
  if (pl > 1.e-6) d.flags->yielded = 1;
  StressRec rec;
  for (int k = 0; k < 6; ++k) rec.s[k] = sig[k];
  rec.rho = rho;
  rec.irho2 = 1.0 / (rho * rho);
  d.srec[i] = rec;
  if (MX) {
    StressRecF rf;
    for (int k = 0; k < 6; ++k) rf.t[k] = (float)(sig[k] * rec.irho2);
    rf.rho = (float)rho;
    rf.pad = 0.0f;
    d.srecf[i] = rf;
  }
  const double vol = o.vol;
  // plastic work heat, Source/ThermalStuct.cpp:14-39 (delta_pl_strain is
  // never reset by the reference, so the last increment keeps heating)
  if (d.pl_heating) {
    double q = d.qpl[i];
    if (d.dpl[i] > 0.0) {
      double dp[6];
      for (int k = 0; k < 6; ++k) dp[k] = d.eplinc[k * np + i] * (1. / dt);
      q = sig[XX] * dp[XX] + 2.0 * sig[XY] * dp[XY] + 2.0 * sig[XZ] * dp[XZ] + sig[YY] * dp[YY] +
          2.0 * sig[YZ] * dp[YZ] + sig[ZZ] * dp[ZZ];
      d.qpl[i] = q;
    }
    d.psen[i] += q * dt;
    e.e_plw = vol * q;
  }
  if (d.thermal) {
    const double Tn = T + dt * d.dTdt[i];
    d.T[i] = Tn;
    e.tmax = Tn;
    e.tmin = Tn;
  } else {
    e.e_int = vol * (Sn[XX] * SR[XX] + 2.0 * Sn[XY] * SR[XY] + 2.0 * Sn[XZ] * SR[XZ] + Sn[YY] * SR[YY] +
                   2.0 * Sn[YZ] * SR[YZ] + Sn[ZZ] * SR[ZZ]);
  }
}

// block partials of the energies, plastic work and temperature range; the
// particles are the block's first kBlock threads (every thread calls this;
// sh: 5 * kBlock / 64 values)
template <bool KIN, bool STRESS>
__device__ inline void rates_sums(const Dev &d, int t, double e_kin, const StressSums &e, double *sh) {
  constexpr int NW = kBlock / 64;
  const int w = threadIdx.x >> 6;
  if (w < NW) {
    const double r[5] = {KIN ? wave_sum(e_kin) : 0.0, STRESS ? wave_sum(e.e_int) : 0.0,
                         STRESS ? wave_sum(e.e_plw) : 0.0, STRESS ? wave_max(e.tmax) : 0.0,
                         STRESS ? wave_min(e.tmin) : 0.0};
    if ((threadIdx.x & 63) == 0)
      for (int q = 0; q < 5; ++q) sh[q * NW + w] = r[q];
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  static_assert(NW == 2, "two wavefronts of particles per block");
  if (KIN) part(d, P_KIN, t) = sh[0] + sh[1];
  if (STRESS) {
    part(d, P_INT, t) = sh[2] + sh[3];
    part(d, P_PLW, t) = sh[4] + sh[5];
    part(d, P_MAXT, t) = fmax(sh[6], sh[7]);
    part(d, P_MINT, t) = fmin(sh[8], sh[9]);
  }
}

// The rate passes' end.  Every lane's partial sums meet in LDS (red: LANES *
// 10 * kBlock values, the staged records' space) and are added in lane order;
// lane 0 of the particle then runs the stress update, lane 1 (with one lane,
// the same) stores the rates and updates the strain.  Both parts' inputs are
// loaded by rates_pre before the tile is staged, so that they arrive during
// the row walk.
template <int LANES>
__device__ inline StressOwn rates_pre(const Dev &d, int buf, int i, int sub, int do_stress) {
  StressOwn o{};
  if (!do_stress || i >= d.n) return o;
  if (sub == 0) o = stress_own(d, buf, i);
  else if (sub == 1)
    for (int k = 0; k < 6; ++k) o.t[k] = d.strain[k * d.npad + i];
  return o;
}
template <bool MX, int LANES, typename R>
__device__ inline void rates_finish(const Dev &d, int i, int sub, R (&v)[10], const StressOwn &o, double dt,
                                    int do_stress, R *red, double *sh) {
  const int lane = threadIdx.x % kBlock;
  if constexpr (LANES > 1) {
    __syncthreads();  // the staged records are read before the sums overwrite them
    for (int c = 0; c < 10; ++c) red[(sub * 10 + c) * kBlock + lane] = v[c];
    __syncthreads();
    if (sub < 2)
      for (int c = 0; c < 10; ++c) {
        R r = red[c * kBlock + lane];
        for (int q = 1; q < LANES; ++q) r += red[(q * 10 + c) * kBlock + lane];
        v[c] = r;
      }
  }
  double e_kin = 0.0;
  StressSums e;
  if (sub < 2 && i < d.n) {
    const bool stress = do_stress && d.group[i] >= 0;
    if (dt < 0) dt = d.flags->dt;
    const double SR[6] = {(double)v[0], (double)v[1], (double)v[2], (double)v[3], (double)v[4], (double)v[5]};
    const double W[3] = {(double)v[6], (double)v[7], (double)v[8]};
    if (sub == LANES - 1 || sub == 1) {
      rates_store(d, i, v);
      if (stress) {
        double strain[6];
        for (int k = 0; k < 6; ++k) strain[k] = LANES == 1 ? d.strain[k * d.npad + i] : o.t[k];
        strain_update(d, i, dt, SR, strain);
      }
    }
    if (sub == 0) {
      e_kin = (double)v[9];
      if (stress) stress_update<MX>(d, i, dt, SR, W, o, e);
    }
  }
  if (do_stress) rates_sums<true, true>(d, blockIdx.x, e_kin, e, sh);
  else rates_sums<true, false>(d, blockIdx.x, e_kin, e, sh);
}

template <int LANES>
__global__ __launch_bounds__(kBlock *LANES) void k_rates_f64(Dev d, int buf, double dt, int do_stress) {
  __shared__ double red[LANES > 1 ? LANES * 10 * kBlock : 1];
  __shared__ double sh[5 * kBlock / 64];
  const int t = xcd_tile(blockIdx.x, gridDim.x), sub = threadIdx.x / kBlock;
  const int i = t * kBlock + (int)(threadIdx.x % kBlock);
  const StressOwn own = rates_pre<LANES>(d, buf, i, sub, do_stress);
  double v[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  if (i < d.n) {
    const HbmJ<false> g{d, buf, i};
    if (d.gc_on) {
      if (d.locking) rates_lane<true, true>(d, buf, i, g, sub, LANES, v);
      else rates_lane<true, false>(d, buf, i, g, sub, LANES, v);
    } else {
      if (d.locking) rates_lane<false, true>(d, buf, i, g, sub, LANES, v);
      else rates_lane<false, false>(d, buf, i, g, sub, LANES, v);
    }
  }
  rates_finish<false, LANES>(d, i, sub, v, own, dt, do_stress, red, sh);
}

// FP64, uniform h: 72 bytes of LDS per staged particle, two blocks per CU;
// the lanes' partial sums reuse the records' space
template <bool GC>
__global__ __launch_bounds__(kBlock *kLanesLds64) __attribute__((amdgpu_waves_per_eu(4))) void k_rates64(Dev d, int buf, double dt, int do_stress) {
  __shared__ double2 rec[kRecRates * kStageMax];
  __shared__ double sc[kStageMax];
  static_assert(2 * kRecRates * kStageMax >= kLanesLds64 * 10 * kBlock, "the partial sums fit the records' space");
  __shared__ double sh[5 * kBlock / 64];
  const int t = xcd_tile(blockIdx.x, gridDim.x), sub = threadIdx.x / kBlock;
  const int i = t * kBlock + (int)(threadIdx.x % kBlock);
  const int U = d.stage_cnt[t];
  const bool on = i < d.n && d.group[i] >= 0;
  const int cnt = on ? d.nnb[i] : 0;
  const double4 xi = d.xh[buf][i], vi = d.vm[i];
  const StressOwn own = rates_pre<kLanesLds64>(d, buf, i, sub, do_stress);
  double v[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  if (U < 0) {
    const HbmRows rows{reinterpret_cast<const int4 *>(d.nbr) + i, d.npad, i};
    if (on)
      rates64_lane<GC>(d, i, i, sub, cnt, xi, vi, RecHbm64<PASS_RATES>::rec_pr(d, buf, i), rows,
                              rows.group(2 * sub), rows.group(2 * sub + 1), RecHbm64<PASS_RATES>{d, buf}, v);
  } else {
    const LdsRows rows{reinterpret_cast<const ushort4 *>(d.nbrl) + i, d.npad, (int)d.selfl[i]};
    const ushort4 a0 = rows.group(2 * sub), b0 = rows.group(2 * sub + 1);
    stage64<kBlock * kLanesLds64, PASS_RATES>(d, buf, t, U, rec, sc, nullptr);
    const RecLds64<PASS_RATES> l{rec, sc, nullptr};
    if (on) rates64_lane<GC>(d, i, rows.own, sub, cnt, xi, vi, l.pr(rows.own), rows, a0, b0, l, v);
  }
  rates_finish<false, kLanesLds64>(d, i, sub, v, own, dt, do_stress, reinterpret_cast<double *>(rec), sh);
}

// CalcRateTensors + RateTensorsReduction in FP32
// (Source/InteractionAlt.cpp:263-479) with the kinetic-energy pair term
// (Source/Domain.cpp:1776-1792).  With c_j = (m_j / rho_j) GK and
// (a, b, g) = c_j e, the sums kept per lane are sum v_x a, v_y b, v_z g
// (diagonal) and the six cross products sum v_x b, v_y a, v_x g, v_z a,
// v_y g, v_z b; strain rate and rotation are their halved sums and
// differences (eps_xy = -(P + Q)/2, w_01 = -(P - Q)/2).  The kinetic term
// carries the lower-index particle's partner mass with a plus sign and the
// higher's with a minus sign; its factor 1/2 is applied at the end.
// v[0..5] strain rate, v[6..8] rotation (w01, w02, w12), v[9] the kinetic sum.
template <int LANES, bool GC, bool STAGED, class Rows, class Rec>
__device__ inline void rates_mx_lane(const Dev &d, int buf, int i, int own, int sub, const Rows &rows,
                                     const Rec &rec, float (&v)[10]) {
  float dxx = 0, dyy = 0, dzz = 0, pxy = 0, qxy = 0, pxz = 0, qxz = 0, pyz = 0, qyz = 0, ek = 0;
  float Li[6];
  own_corr<GC>(d, i, Li);
  const float4 xi = d.xhf[buf][i], vi = d.vmf[i];
  const float pri = d.prf[i], mneg = -vi.w;
  const GkF k = gk_consts((float)d.xh[buf][i].w, d.dim);
  walk_groups<LANES>(rows, d.nnb[i], sub, rows.self(), rows.group(2 * sub), rows.group(2 * sub + 1), [&](const typename Rows::G &c) {
    float4 X[4], V[4];
    float P[4];
    int l[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      l[u] = entry(c, u);
      rec.load(l[u], X[u], V[u]);
      P[u] = rec.pr(l[u]);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float dx = xi.x - X[u].x, dy = xi.y - X[u].y, dz = xi.z - X[u].z;
      const float GK = gk_f(dx * dx + dy * dy + dz * dz, k);
      const float vx = vi.x - V[u].x, vy = vi.y - V[u].y, vz = vi.z - V[u].z;
      const float cj = X[u].w * GK;
      float ex, ey, ez;
      corr_dir<GC>(Li, dx, dy, dz, ex, ey, ez);
      const float a = cj * ex, b = cj * ey, g = cj * ez;
      dxx = fmaf(vx, a, dxx);
      dyy = fmaf(vy, b, dyy);
      dzz = fmaf(vz, g, dzz);
      pxy = fmaf(vx, b, pxy);
      qxy = fmaf(vy, a, qxy);
      pxz = fmaf(vx, g, pxz);
      qxz = fmaf(vz, a, qxz);
      pyz = fmaf(vy, g, pyz);
      qyz = fmaf(vz, b, qyz);
      // staged positions follow particle index order
      const bool lo = STAGED ? own < l[u] : i < l[u];
      const float ms = lo ? V[u].w : mneg;
      ek = fmaf(ms * (pri + P[u]), GK * (vx * dx + vy * dy + vz * dz), ek);
    }
  });
  v[XX] = -dxx;
  v[YY] = -dyy;
  v[ZZ] = -dzz;
  v[XY] = -0.5f * (pxy + qxy);
  v[XZ] = -0.5f * (pxz + qxz);
  v[YZ] = -0.5f * (pyz + qyz);
  v[6] = -0.5f * (pxy - qxy);
  v[7] = -0.5f * (pxz - qxz);
  v[8] = -0.5f * (pyz - qyz);
  v[9] = 0.5f * ek;
}

template <int LANES, bool GC>
__global__ __launch_bounds__(kBlock *LANES) void k_rates_mx(Dev d, int buf, double dt, int do_stress) {
  __shared__ float4 lx[2 * (kStageMax + 1)];
  __shared__ float lp[kStageMax + 1];
  float4 *lv = lx + kStageMax + 1;
  static_assert(8 * (kStageMax + 1) >= LANES * 10 * kBlock, "the partial sums fit the records' space");
  __shared__ double sh[5 * kBlock / 64];
  const int t = xcd_tile(blockIdx.x, gridDim.x), sub = threadIdx.x / kBlock;
  const int i = t * kBlock + (int)(threadIdx.x % kBlock);
  const int U = d.stage_cnt[t];
  const StressOwn own = rates_pre<LANES>(d, buf, i, sub, do_stress);
  float v[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  if (U < 0) {
    if (i < d.n && d.group[i] >= 0) {
      const HbmRows rows{reinterpret_cast<const int4 *>(d.nbr) + i, d.npad, i};
      rates_mx_lane<LANES, GC, false>(d, buf, i, i, sub, rows, XvHbm{d.xhf[buf], d.vmf, d.prf}, v);
    }
  } else {
    stage_xv<kBlock * LANES>(d, t, U, d.xhf[buf], lx, lv, lp);
    if (i < d.n && d.group[i] >= 0) {
      const LdsRows rows{reinterpret_cast<const ushort4 *>(d.nbrl) + i, d.npad, (int)d.selfl[i]};
      rates_mx_lane<LANES, GC, true>(d, buf, i, d.selfl[i], sub, rows, XvLds{lx, lv, lp}, v);
    }
  }
  rates_finish<true, LANES>(d, i, sub, v, own, dt, do_stress, reinterpret_cast<float *>(lx), sh);
}

// the stress update alone (single-pass evaluations; the step above kFuseTiles tiles)
template <bool MX>
WF_KERNEL void k_stress(Dev d, int buf, double dt) {
  if (dt < 0) dt = d.flags->dt;
  __shared__ double sh[5 * kBlock / 64];
  const int i = blockIdx.x * kBlock + threadIdx.x;
  const long long np = d.npad;
  StressSums e;
  if (i < d.n && d.group[i] >= 0) {
    double SR[6], W[3];
    for (int k = 0; k < 6; ++k) SR[k] = d.sr[k * np + i];
    for (int k = 0; k < 3; ++k) W[k] = d.rr[k * np + i];
    double strain[6];
    for (int k = 0; k < 6; ++k) strain[k] = d.strain[k * np + i];
    strain_update(d, i, dt, SR, strain);
    stress_update<MX>(d, i, dt, SR, W, stress_own(d, buf, i), e);
  }
  rates_sums<false, true>(d, blockIdx.x, 0.0, e, sh);
}

// The stress update runs inside the rate kernel up to about one tile per CU:
// there a launch costs more than what the update's dependent chain (return
// map, powers) adds to each block.  In large models a kernel of its own keeps
// more of those chains in flight.  Whole yielding steps, fused against apart, us
// (mixed; FP64; FP64 with damage):
//   9k     79  81    81  83    79  82
//   41k    95  99   109 113   111 115
//   95k   116 120   156 160   162 166
//   193k  165 166   224 222   235 230
//   954k  625 616   954 918   964 908
// so the line lies on the safe side: fused is 3 % faster up to about 100k
// particles.
constexpr int kFuseTiles = 320;
bool launch_rates(const Dev &d, hipStream_t st, int buf, double dt, int do_stress) {
  if (d.ntiles > kFuseTiles) do_stress = 0;
  if (d.mixed) {
    WF_LANES_GC_SWITCH(d.lanes_mx, d.gc_on, k_rates_mx, d, buf, dt, do_stress)
  } else {
    if (d.lds64) {
      gc_switch(d.gc_on, [&](auto gc) {
        k_rates64<decltype(gc)::value><<<nblk(d.n), kBlock * kLanesLds64, 0, st>>>(d, buf, dt, do_stress);
      });
    } else {
      WF_LANES_SWITCH(d.lanes_f64, k_rates_f64, d, buf, dt, do_stress)
    }
  }
  return do_stress != 0;
}

void launch_stress(const Dev &d, hipStream_t st, int buf, double dt) {
  if (d.mixed)
    k_stress<true><<<d.nblocks, kBlock, 0, st>>>(d, buf, dt);
  else
    k_stress<false><<<d.nblocks, kBlock, 0, st>>>(d, buf, dt);
}

// ---------------------------------------------------------------------------
// conduction (CalcTempInc, Source/Thermal.cpp:53-219) + convection
// (CalcConvHeat, :339-389) + thermal expansion (Source/ThermalStuct.cpp:7-12)
// The reference credits temp[first] += m and temp[second] -= m with m built
// from the second particle's m/rho (first, second: see thermal_key).  FP64 in
// both precision modes.
//
// The gather kernel (one lane per particle; positions, T, m/rho, cells and
// indices of each neighbour from HBM, the cells' order by integer divisions)
// took 211 us at 370k particles, bound by the latency of its dependent loads.
// From the tile's LDS copy (48 bytes per staged particle) 64 us with two lanes
// and three blocks per CU, 79 us with four lanes (two blocks, register bound).
// The gather remains for smoothing lengths that differ within a material.

// the particle's own side after the gather: convection, sources, dT/dt, the
// thermal strain rate; returns the internal energy rate and the contact heat
// totals' terms (Source/Thermal.cpp:194-210)
__device__ inline double3 thermal_own(const Dev &d, int buf, int i, double temp) {
  const long long np = d.npad;
  const DevMat &M = d.mats[d.mat[i]];
  const double rho = d.rho[buf][i], m = d.vm[i].w, Ti = d.T[i], voli = d.vol[buf][i];
  double qconv = d.qconv[i];
  if (d.thbc[i] == 1) {
    // (m/rho)^(2/3), (m/rho)^(1/3) in plane strain (Source/Thermal.cpp:354-366)
    const double dS2 = pow(m / rho, d.dim == 2 ? 1.0 / 3.0 : 2.0 / 3.0);
    qconv = rho * d.hconv[i] * dS2 * (d.tinf[i] - Ti) / m;
    d.qconv[i] = qconv;
  }
  const double f = 1. / (rho * M.cp_T);
  const double qc = d.heat_cond ? d.qcont[i] : 0.0;
  double dTdt = f * (temp + qconv + d.qsrc[i] + d.qpl[i] * d.pl_frac + qc);
  if (d.heat_fric) dTdt += f * d.qfric[i];
  d.dTdt[i] = dTdt;
  double3 e = make_double3(0.0, 0.0, 0.0);
  if (d.qfric) {
    e.y = d.qfric[i] * m / rho;
    e.z = qc * m / rho;
  }
  double SR[6];
  for (int k = 0; k < 6; ++k) SR[k] = d.sr[k * np + i];
  const double ex = M.th_exp * dTdt;
  for (int k = 0; k < 3; ++k) {
    SR[k] += ex;
    d.sr[k * np + i] = SR[k];
  }
  double S[6];
  for (int k = 0; k < 6; ++k) S[k] = d.S[k * np + i];
  e.x = voli * (S[XX] * SR[XX] + 2.0 * S[XY] * SR[XY] + 2.0 * S[XZ] * SR[XZ] + S[YY] * SR[YY] +
                2.0 * S[YZ] * SR[YZ] + S[ZZ] * SR[ZZ]);
  return e;
}
__device__ inline void thermal_sums(const Dev &d, const double3 &e, int t, double *sh) {
  const double r0 = block_reduce<0>(e.x, sh);
  if (threadIdx.x == 0) part(d, P_INT, t) = r0;
  if (d.qfric) {
    const double r1 = block_reduce<0>(e.y, sh);
    const double r2 = block_reduce<0>(e.z, sh);
    if (threadIdx.x == 0) {
      part(d, P_FRW, t) = r1;
      part(d, P_CHC, t) = r2;
    }
  }
}
// the conductivity factor of a pair (both particles of one material)
__device__ inline double pair_kk(const DevMat &M) { return 4. * (M.k_T * M.k_T) / (M.k_T + M.k_T); }

WF_KERNEL void k_thermal(Dev d, int buf) {
  __shared__ double sh[kBlock / 64];
  const int t = xcd_tile(blockIdx.x, gridDim.x);
  const int i = t * kBlock + threadIdx.x;
  double3 e = make_double3(0.0, 0.0, 0.0);
  if (i < d.n && d.group[i] >= 0) {
    const double4 xi = d.xh[buf][i];
    const double Ti = d.T[i], voli = d.vol[buf][i], kk = pair_kk(d.mats[d.mat[i]]);
    const long long ki = d.tkey[i];
    double temp = 0.0;
    const KernH kh = kern_h(xi.w, d.dim);
    const int cnt = d.nnb[i];
    for (int k = 0; k < cnt; ++k) {
      const int j = d.nbr[nb_slot(d.npad, k, i)];
      const double4 xj = d.xh[buf][j];
      const double dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
      const double r2 = dx * dx + dy * dy + dz * dz;
      const double GK = grad_kernel_r2(r2, pair_h(kh, xi.w, xj.w));
      const double vsec = d.tkey[j] > ki ? d.vol[buf][j] : voli;
      // dot(x_ij, GK x_ij) / |x_ij|^2 = GK
      temp += vsec * kk * (Ti - d.T[j]) * GK;
    }
    e = thermal_own(d, buf, i, temp);
  }
  thermal_sums(d, e, t, sh);
}

// records of the conduction gather: (x, y), (z, T), (m/rho, key)
struct HeatLds {
  const double2 *r;
  __device__ void load(int p, double &x, double &y, double &z, double &T, double &vol, long long &key) const {
    const double2 a = r[p], b = r[kStageMax + p], c = r[2 * kStageMax + p];
    x = a.x, y = a.y, z = b.x, T = b.y, vol = c.x, key = __double_as_longlong(c.y);
  }
};
struct HeatHbm {
  const Dev &d;
  const int buf;
  __device__ void load(int j, double &x, double &y, double &z, double &T, double &vol, long long &key) const {
    const double4 a = d.xh[buf][j];
    x = a.x, y = a.y, z = a.z, T = d.T[j], vol = d.vol[buf][j], key = d.tkey[j];
  }
};
constexpr int kLanesHeat = 2;
template <class Rows, class Rec>
__device__ inline double heat_lane(const Dev &d, int sub, int cnt, const double4 &xi, double Ti, double voli,
                                   long long ki, const Rows &rows, typename Rows::G a0, typename Rows::G b0,
                                   const Rec &rec) {
  double s = 0.0;
  const GkD k = gk_consts64(xi.w, d.dim);
  walk_groups<kLanesHeat>(rows, cnt, sub, rows.self(), a0, b0, [&](const typename Rows::G &c) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      double x, y, z, T, vol;
      long long key;
      rec.load(entry(c, u), x, y, z, T, vol, key);
      const double dx = xi.x - x, dy = xi.y - y, dz = xi.z - z;
      const double GK = gk_d(dx * dx + dy * dy + dz * dz, k);
      s = fma((key > ki ? vol : voli) * (Ti - T), GK, s);
      if (u & 1) __builtin_amdgcn_sched_barrier(0);
    }
  });
  return s;
}
__global__ __launch_bounds__(kBlock *kLanesHeat) void k_thermal_lds(Dev d, int buf) {
  constexpr int NT = kBlock * kLanesHeat;
  __shared__ double2 rec[3 * kStageMax];
  __shared__ double red[(kLanesHeat - 1) * kBlock];
  __shared__ double sh[NT / 64];
  const int t = xcd_tile(blockIdx.x, gridDim.x), sub = threadIdx.x / kBlock;
  const int i = t * kBlock + (int)(threadIdx.x % kBlock);
  const int U = d.stage_cnt[t];
  const bool on = i < d.n && d.group[i] >= 0;
  const int cnt = on ? d.nnb[i] : 0;
  const double4 xi = d.xh[buf][i];
  const double Ti = d.T[i], voli = d.vol[buf][i];
  const long long ki = d.tkey[i];
  double s[1] = {0.0};
  if (U < 0) {
    const HbmRows rows{reinterpret_cast<const int4 *>(d.nbr) + i, d.npad, i};
    if (on)
      s[0] = heat_lane(d, sub, cnt, xi, Ti, voli, ki, rows, rows.group(2 * sub), rows.group(2 * sub + 1),
                       HeatHbm{d, buf});
  } else {
    const LdsRows rows{reinterpret_cast<const ushort4 *>(d.nbrl) + i, d.npad, (int)d.selfl[i]};
    const ushort4 a0 = rows.group(2 * sub), b0 = rows.group(2 * sub + 1);
    const HeatHbm h{d, buf};
    stage_set<NT>(d.stage, t, U, [&](int p, int j) {
      double x, y, z, T, vol;
      long long key;
      h.load(j, x, y, z, T, vol, key);
      rec[p] = make_double2(x, y);
      rec[kStageMax + p] = make_double2(z, T);
      rec[2 * kStageMax + p] = make_double2(vol, __longlong_as_double(key));
    });
    if (on) s[0] = heat_lane(d, sub, cnt, xi, Ti, voli, ki, rows, a0, b0, HeatLds{rec});
  }
  combine_lanes<kLanesHeat>(s, red);
  __builtin_amdgcn_sched_barrier(0);
  double3 e = make_double3(0.0, 0.0, 0.0);
  // (no pairs, no factor: a conductivity of 0 makes it 0/0)
  if (on && sub == 0) e = thermal_own(d, buf, i, cnt > 0 ? pair_kk(d.mats[d.mat[i]]) * s[0] : 0.0);
  thermal_sums(d, e, t, sh);
}

void launch_thermal(const Dev &d, hipStream_t st, int buf) {
  if (d.h_uni) k_thermal_lds<<<d.nblocks, kBlock * kLanesHeat, 0, st>>>(d, buf);
  else k_thermal<<<d.nblocks, kBlock, 0, st>>>(d, buf);
}

// ---------------------------------------------------------------------------
// end of step: fixed-order reduction of the block partials, scalar updates,
// reaction history, and the end-of-step half of the neighbour schedule.
// One block per active slot sums that slot's partials (each thread its
// blocks in order, four loads in flight, then the wavefront butterfly and
// the wavefronts in order), so the slots reduce in parallel across CUs; the
// block that finishes last (a ticket counter, reset by that block for the
// next step) then applies them with one thread.

struct FinList {
  int n;
  int slot[P_COUNT];
  int op[P_COUNT];  // 0 sum, 1 max, 2 min
};

__device__ inline double fin_op(int op, double v, double x) {
  return op == 0 ? v + x : (op == 1 ? fmax(v, x) : fmin(v, x));
}

// val: the reduced slots, in the list's order
__device__ void fin_apply(const Dev &d, double dt, const FinList &L, const double *val) {
  if (dt < 0) dt = d.flags->dt;
  DevFlags *f = d.flags;
  const long long step = f->step;
  const long long slot = step % d.hist_cap;
  double e_kin = 0.0, e_int = 0.0, plw = 0.0, tmax = 0.0, tmin = 0.0, cfsum = 0.0, creact = 0.0, extw = 0.0;
  for (int k = 0; k < L.n; ++k) {
    const int s = L.slot[k];
    const double r = val[k];
    if (s == P_KIN) e_kin = r;
    if (s == P_INT) e_int = r;
    if (s == P_PLW) plw = r;
    if (s == P_MAXT) tmax = r;
    if (s == P_MINT) tmin = r;
    if (s >= P_REACT && s < P_CFORCE) d.react_hist[slot * kMaxZones * 3 + (s - P_REACT)] = r;
    if (s >= P_CFORCE && s < P_CFSUM) d.cf_hist[slot * kMaxMesh * 3 + (s - P_CFORCE)] = r;
    if (s == P_CFSUM) cfsum = r;
    if (s == P_CREACT) creact = r;
    if (s == P_EXTW) extw = r;
    if (s == P_FRW) d.scalars[S_FRW] += r * dt;
    if (s == P_CHC) d.scalars[S_CHC] += r * dt;
  }
  if (d.contact) {
    d.scalars[S_CFSUM] = cfsum;
    d.scalars[S_CREACT] = creact;
    d.scalars[S_EXTW] += extw;
  }
  d.scalars[S_KIN] += e_kin * dt;
  d.scalars[S_INT] += e_int * dt;
  if (d.pl_heating) d.scalars[S_PLW] += plw * dt;
  if (d.thermal) {
    d.scalars[S_MAXT] = fmax(0.0, tmax);
    d.scalars[S_MINT] = fmin(1000.0, tmin);
  }
  if (!isfinite(e_int)) f->nan = 1;
  if (f->step_yield) {
    if (f->ts_i == f->ts_nb_inc - 1) f->cleared = 1;
    f->ts_i++;
    if (f->ts_i > f->ts_nb_inc - 1) f->ts_i = 0;
  }
  f->step = step + 1;
  f->time += dt;
}

// TriMesh::Update of mesh m by one block (Source/Mesh.cpp:273-296): node
// velocity m_v + m_w x node at the node's position before it moves, nodes
// move with it, element normals and plane coefficients are recomputed from
// the winding, particles take the mean node velocity.  drift: the rigid
// particles' drift with their old velocities first (the reference's loop
// covers them).
__device__ inline void mesh_update(const Dev &d, int m, double dt, int drift) {
  const double4 mv = d.mv[m], mw = d.mw[m];
  const int n0 = d.mesh_node0[m], nn = d.mesh_nnode[m];
  for (int k = threadIdx.x; k < nn; k += blockDim.x) {
    double4 p = d.node[n0 + k];
    const double wp[3] = {mw.y * p.z - mw.z * p.y, mw.z * p.x - mw.x * p.z, mw.x * p.y - mw.y * p.x};
    const double4 nv = make_double4(mv.x + wp[0], mv.y + wp[1], mv.z + wp[2], 0.0);
    p.x += nv.x * dt;
    p.y += nv.y * dt;
    p.z += nv.z * dt;
    d.node[n0 + k] = p;
    d.nodev[n0 + k] = nv;
  }
  __syncthreads();
  const int e0 = d.mesh_elem0[m], ne = d.mesh_nelem[m];
  for (int e = threadIdx.x; e < ne; e += blockDim.x) {
    const int4 el = d.elem[e0 + e];
    if (drift) {
      double4 x = d.rx[e0 + e];
      const double4 v = d.rv[e0 + e];
      x.x += v.x * dt;
      x.y += v.y * dt;
      x.z += v.z * dt;
      d.rx[e0 + e] = x;
    }
    const double4 a = d.node[el.x], b = d.node[el.y], c = d.node[el.z];
    const double u[3] = {b.x - a.x, b.y - a.y, b.z - a.z}, v[3] = {c.x - a.x, c.y - a.y, c.z - a.z};
    double w[3];
    cross_d(u, v, w);
    const double nw = sqrt(w[0] * w[0] + w[1] * w[1] + w[2] * w[2]);
    const double n[3] = {w[0] / nw, w[1] / nw, w[2] / nw};
    const double4 pf = el.w == 0 ? a : (el.w == 1 ? b : c);
    const double pp = pf.x * n[0] + pf.y * n[1] + pf.z * n[2];
    d.enorm[e0 + e] = make_double4(n[0], n[1], n[2], pp);
    const double4 va = d.nodev[el.x], vb = d.nodev[el.y], vc = d.nodev[el.z];
    const double vm = ((0.0 + va.x) + vb.x) + vc.x;
    const double vn = ((0.0 + va.y) + vb.y) + vc.y;
    const double vo = ((0.0 + va.z) + vb.z) + vc.z;
    d.rv[e0 + e] = make_double4(vm / 3, vn / 3, vo / 3, 0.0);
  }
}

// blocks [0, L.n): the slots; then one block per rigid mesh.  The handed-over
// sums are written through and loaded by as many threads at once: with
// __threadfence() and one thread loading them in turn the kernel took 6-12 us,
// 5.8 us at 4.5k particles and 16 with two meshes of 2,048 triangles now; the
// meshes' update was a launch of its own of 10-15 us and the drift
// one of 4.6 us.
constexpr int kFinThreads = 1024;
__global__ __launch_bounds__(kFinThreads) void k_finalize(Dev d, double dt, FinList L, int drift) {
  __shared__ double sh[kFinThreads / 64];
  __shared__ double val[P_COUNT];
  __shared__ int last;
  if ((int)blockIdx.x >= L.n) {
    mesh_update(d, blockIdx.x - L.n, dt < 0 ? d.flags->dt : dt, drift);
    return;
  }
  const int s = L.slot[blockIdx.x], op = L.op[blockIdx.x];
  const int nb = d.nblocks;
  double v = op == 0 ? 0.0 : (op == 1 ? -INFINITY : INFINITY);
  for (int b = threadIdx.x; b < nb; b += 4 * blockDim.x) {
    double x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int bu = b + u * (int)blockDim.x;
      x[u] = bu < nb ? part(d, s, bu) : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (b + u * (int)blockDim.x < nb) v = fin_op(op, v, x[u]);
  }
  double r;
  if (op == 0) r = block_reduce<0>(v, sh);
  else if (op == 1) r = block_reduce<1>(v, sh);
  else r = block_reduce<2>(v, sh);
  if (threadIdx.x == 0) {
    put_agent(&d.fin[s], r);
    stores_done();
    last = atomicAdd(&d.flags->fin_ticket, 1u) == (unsigned)(L.n - 1);
  }
  __syncthreads();
  if (!last) return;
  if ((int)threadIdx.x < L.n) val[threadIdx.x] = get_agent(&d.fin[L.slot[threadIdx.x]]);
  __syncthreads();
  if (threadIdx.x != 0) return;
  fin_apply(d, dt, L, val);
  d.flags->fin_ticket = 0;
}

void launch_finalize(const Dev &d, hipStream_t st, double dt, int nz, int drift) {
  FinList L{};
  auto add = [&](int s, int op) {
    L.slot[L.n] = s;
    L.op[L.n] = op;
    ++L.n;
  };
  add(P_INT, 0);
  add(P_KIN, 0);
  if (d.pl_heating) add(P_PLW, 0);
  if (d.thermal) {
    add(P_MAXT, 1);
    add(P_MINT, 2);
  }
  for (int s = P_REACT; s < P_REACT + 3 * nz; ++s) add(s, 0);
  if (d.contact) {
    for (int s = P_CFORCE; s < P_CFORCE + 3 * d.nmesh; ++s) add(s, 0);
    add(P_CFSUM, 0);
    add(P_CREACT, 0);
    add(P_EXTW, 0);
    if (d.thermal && d.qfric) {
      add(P_FRW, 0);
      add(P_CHC, 0);
    }
  }
  k_finalize<<<L.n + (d.contact ? d.nmesh : 0), kFinThreads, 0, st>>>(d, dt, L, drift);
}

// ---------------------------------------------------------------------------
// rigid contact planes: free-surface detection (Domain::CalculateSurface,
// Source/Domain.cpp:1415-1491), contact pairs (AllocateNbPair's contact
// branch + ContactNbSearch, Source/Neighbour.cpp:375-396,
// Source/Contact.cpp:57-132), the Wang penalty force with Coulomb friction
// (Source/Contact_Wang.cpp:15-348) and the rigid-body motion of the planes
// (TriMesh::Update, Source/Mesh.cpp:273-296; UpdateContactParticles,
// Source/Contact.cpp:41-55).  FP64 in both precision modes.


// After a neighbour build.  A particle was on the free surface (ID 1) when
// the search ran; the new surface test then uses the new rows.  Contact
// partners are the rigid particles, in index order, of an adjacent cell
// closer than h_i + h_r, for particles on the surface before and after.
// setup = 1: the search before the first step only sets the surface.
// setup = 2: with damage, every step after the search (CalculateSurface(1),
// Source/SolverLeapfrog.cpp:204-206): the surface ids only.
//
// A block takes P particles: the first P threads test their surface and walk
// up to kSurfOwn rigid candidates each; particles with more are then searched
// by whole wavefronts, 64 candidates at a time.  Coarse rigid surfaces put
// thousands of candidates into a particle's 27 cells: one lane walking them
// took 394 us per search of a 1.3k-particle specimen between two planes of
// 2,048 triangles, now 59 us.  Wavefronts for every surface particle were
// slower where candidates are few (a forging of 370k particles, 234 against
// 74 us per search; 601k in 64 specimens 432 against 159).
constexpr int kSurfOwn = 256;
// the ranges of binned rigid particles in the 27 cells around cell ci: column
// after column, f(first, end)
template <class F>
__device__ inline void for_rigid_ranges(const Dev &d, int ci, F &&f) {
  const int gz = d.cellno[2], gy = d.cellno[1], gx = d.cellno[0];
  const int cz = ci % gz, cy = (ci / gz) % gy, cx = ci / (gz * gy);
  for (int ax = cx - 1; ax <= cx + 1; ++ax) {
    if (ax < 0 || ax >= gx) continue;
    for (int ay = cy - 1; ay <= cy + 1; ++ay) {
      if (ay < 0 || ay >= gy) continue;
      const int c0 = (ax * gy + ay) * gz;
      f(d.rstart[c0 + (cz > 0 ? cz - 1 : 0)], d.rstart[c0 + (cz + 1 < gz ? cz + 1 : gz - 1) + 1]);
    }
  }
}
__device__ inline bool rigid_near(const double4 &x, const double4 &xr) {
  const double dx = x.x - xr.x, dy = x.y - xr.y, dz = x.z - xr.z;
  return sqrt(dx * dx + dy * dy + dz * dz) < x.w + xr.w;
}
template <int P>
WF_KERNEL void k_surface(Dev d, int cur, int setup) {
  if (setup != 2 && !d.flags->do_search) return;
  __shared__ int need[P];
  __shared__ int nneed;
  __shared__ int found[kBlock / 64][kMaxContact];
  const long long np = d.npad;
  const int tid = threadIdx.x;
  if (tid == 0) nneed = 0;
  __syncthreads();
  const int i = blockIdx.x * P + tid;
  if (tid < P && i < d.n) {
    const int old_surf = d.id[i] == 1;
    const double4 xi = d.xh[cur][i];
    double nx = 0.0, ny = 0.0, nz = 0.0;
    const int cnt = d.nnb[i];
    // a free-surface particle has at most 46 neighbours (12 in 2D,
    // Source/Domain.cpp:1472-1474); with more the test fails whatever the
    // normal, so the row is not walked.  Otherwise the row's groups of four
    // entries, their gathers issued together; the sum runs over the entries
    // in row order
    const int nb_max = d.dim == 2 ? 12 : 46;
    const int4 *row = reinterpret_cast<const int4 *>(d.nbr) + i;
    for (int g = 0; cnt <= nb_max && 4 * g < cnt; ++g) {
      const int4 e = row[(long long)g * np];
      const int jj[4] = {e.x, e.y, e.z, e.w};
      double4 xj[4];
      double mj[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        xj[u] = d.xh[cur][jj[u]];
        mj[u] = d.pmass[jj[u]];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (4 * g + u >= cnt) break;
        nx += mj[u] * (xi.x - xj[u].x);
        ny += mj[u] * (xi.y - xj[u].y);
        nz += mj[u] * (xi.z - xj[u].z);
      }
    }
    const double f = 1. / d.totmass;
    nx *= f;
    ny *= f;
    nz *= f;
    const int surf = cnt <= nb_max && sqrt(nx * nx + ny * ny + nz * nz) >= 0.25 * xi.w;
    d.id[i] = surf ? 1 : d.id_orig[i];
    if (setup != 2) {
      // few candidates: the particle's own lane takes them; many: a wavefront
      int c = 0, cand = 0;
      if (!setup && old_surf && surf) {
        for_rigid_ranges(d, d.cell[i], [&](int p0, int p1) { cand += p1 - p0; });
        if (cand > kSurfOwn) {
          need[atomicAdd(&nneed, 1)] = i;
        } else if (cand > 0) {
          for_rigid_ranges(d, d.cell[i], [&](int p0, int p1) {
            for (int p = p0; p < p1; ++p) {
              const int r = d.rsorted[p];
              if (!rigid_near(xi, d.rx[r])) continue;
              if (c < kMaxContact) {
                int q = c;
                while (q > 0 && d.cidx[(long long)(q - 1) * np + i] > r) {
                  d.cidx[(long long)q * np + i] = d.cidx[(long long)(q - 1) * np + i];
                  --q;
                }
                d.cidx[(long long)q * np + i] = r;
              }
              ++c;
            }
          });
          if (c > kMaxContact) d.flags->overflow = 1;
        }
      }
      if (cand <= kSurfOwn) d.ccnt[i] = c < kMaxContact ? c : kMaxContact;
    }
  }
  if (setup) return;
  __syncthreads();
  // ContactNbSearch: the rigid particles of the 27 cells around the
  // particle's own (binned by k_cell_hist / k_scatter at this search),
  // |x_ij| < h_i + h_r; partners are kept in rigid-particle index order
  const int lane = tid & 63, w = tid >> 6;
  volatile int *fw = found[w];
  const int gz = d.cellno[2], gy = d.cellno[1], gx = d.cellno[0];
  for (int q = w; q < nneed; q += kBlock / 64) {
    const int k = need[q];
    const double4 xk = d.xh[cur][k];
    const int ck = d.cell[k];
    const int cz = ck % gz, cy = (ck / gz) % gy, cx = ck / (gz * gy);
    // lane c < 9: column c's range of binned rigid particles
    int lo = 0, hi = 0;
    if (lane < 9) {
      const int ax = cx + lane / 3 - 1, ay = cy + lane % 3 - 1;
      if (ax >= 0 && ax < gx && ay >= 0 && ay < gy) {
        const int c0 = (ax * gy + ay) * gz;
        lo = d.rstart[c0 + (cz > 0 ? cz - 1 : 0)];
        hi = d.rstart[c0 + (cz + 1 < gz ? cz + 1 : gz - 1) + 1];
      }
    }
    int c = 0;
    unsigned long long cols = __ballot(hi > lo);
    while (cols) {
      const int col = __ffsll((long long)cols) - 1;
      cols &= cols - 1;
      const int p0 = __shfl(lo, col, 64), p1 = __shfl(hi, col, 64);
      for (int base = p0; base < p1; base += 64) {
        const int p = base + lane;
        bool in = false;
        int r = 0;
        if (p < p1) {
          r = d.rsorted[p];
          in = rigid_near(xk, d.rx[r]);
        }
        const unsigned long long m = __ballot(in);
        const int at = c + __popcll(m & ((1ull << lane) - 1));
        if (in && at < kMaxContact) fw[at] = r;
        c += __popcll(m);
      }
    }
    __builtin_amdgcn_wave_barrier();
    const int kept = c < kMaxContact ? c : kMaxContact;
    if (lane < kept) {
      const int r = fw[lane];
      int rank = 0;
      for (int o = 0; o < kept; ++o) rank += fw[o] < r ? 1 : 0;
      d.cidx[(long long)rank * np + k] = r;
    }
    __builtin_amdgcn_wave_barrier();
    if (lane == 0) {
      d.ccnt[k] = kept;
      if (c > kMaxContact) d.flags->overflow = 1;
    }
  }
}

// the planes' velocities alone, for a step run in parts
WF_KERNEL void k_rigid_bc(Dev d, BcTable bc) { rigid_bc(d, bc, blockIdx.x * kBlock + threadIdx.x); }

// Wang contact force of each particle over its partners, in order
WF_KERNEL void k_contact(Dev d, int cur, double dt) {
  if (dt < 0) dt = d.flags->dt;
  __shared__ double sh[kBlock / 64];
  const int i = blockIdx.x * kBlock + threadIdx.x;
  double cfm[kMaxMesh][3];
  for (int m = 0; m < kMaxMesh; ++m) cfm[m][0] = cfm[m][1] = cfm[m][2] = 0.0;
  double cfsum = 0.0, creact = 0.0, extw = 0.0, fts = INFINITY;
  if (i < d.n) {
    double cf[3] = {0, 0, 0};
    double qf = 0.0, fh = 0.0, cs = 0.0, qc = 0.0;
    double cfi[kMaxMesh][3];  // this particle's contact force per mesh
    for (int m = 0; m < kMaxMesh; ++m) cfi[m][0] = cfi[m][1] = cfi[m][2] = 0.0;
    const int cnt = d.ccnt[i];
    if (cnt > 0) {
      const double4 x4 = d.xh[cur][i];
      const double4 v4 = d.vm[i];
      double4 a4 = d.acc[i];
      const double x[3] = {x4.x, x4.y, x4.z}, v[3] = {v4.x, v4.y, v4.z};
      double a[3] = {a4.x, a4.y, a4.z};
      const double h = x4.w, m1 = v4.w;
      const DevMat &Mi = d.mats[d.mat[i]];
      double fr_sta = Mi.fr_sta >= 0.0 ? Mi.fr_sta : d.fr_sta;
      double fr_dyn = Mi.fr_sta >= 0.0 ? Mi.fr_dyn : d.fr_dyn;
      // friction_function Linear (Source/Contact_Wang.cpp:241-244)
      if (d.fric_linear) fr_sta = fr_dyn = d.fr_m * d.T[i] + d.fr_b;
      for (int q = 0; q < cnt; ++q) {
        const int r = d.cidx[(long long)q * d.npad + i];
        const int mi = d.rmesh[r];
        const double4 en = d.enorm[r];
        const double n2[3] = {en.x, en.y, en.z};
        const double4 v24 = d.rv[r];
        const double v2[3] = {v24.x, v24.y, v24.z};
        const double delta_ = -(n2[0] * (v[0] - v2[0]) + n2[1] * (v[1] - v2[1]) + n2[2] * (v[2] - v2[2]));
        double xp[3];
        for (int k = 0; k < 3; ++k) xp[k] = x[k] + v[k] * dt + a[k] * dt * dt / 2.0;
        const double dist = (n2[0] * xp[0] + n2[1] * xp[1] + n2[2] * xp[2]) - en.w;
        if (!(dist < h)) continue;
        double qj[3];
        for (int k = 0; k < 3; ++k) qj[k] = x[k] - dist * n2[k];
        const int4 el = d.elem[r];
        const int nd[3] = {el.x, el.y, el.z};
        bool inside = true;
        for (int ii = 0; ii < 3 && inside; ++ii) {
          const int jj = ii + 1 > 2 ? 0 : ii + 1;
          const double4 ni = d.node[nd[ii]], nj = d.node[nd[jj]];
          const double ea[3] = {nj.x - ni.x, nj.y - ni.y, nj.z - ni.z};
          const double eb[3] = {qj[0] - ni.x, qj[1] - ni.y, qj[2] - ni.z};
          double c[3];
          cross_d(ea, eb, c);
          if (c[0] * n2[0] + c[1] * n2[1] + c[2] * n2[2] < 0.0) inside = false;
        }
        if (!inside) continue;
        const double delta = h - dist;
        const double kij = 2.0 * m1 / (dt * dt);
        const double omega = sqrt(kij / m1);
        const double psi = 2. * m1 * omega * d.dfac;
        for (int k = 0; k < 3; ++k) cf[k] = (kij * delta - psi * delta_) * n2[k];
        {
          // dt_fext on the normal force (Source/Contact_Wang.cpp:226-233);
          // Domain::min_force_ts takes the least below 1000
          const double nv = sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
          const double nc = sqrt(cf[0] * cf[0] + cf[1] * cf[1] + cf[2] * cf[2]);
          const double dt_fext = 1. * (m1 * 2. * nv / nc);
          if (dt_fext < 1000. && dt_fext < fts) fts = dt_fext;
        }
        for (int k = 0; k < 3; ++k) a[k] += cf[k] / m1;
        // Fraser 3-119: the contact area of the particle, formed whenever a
        // contact heat branch (the only readers, which divide by it) is on
        const double dens = d.rho[cur][i];
        const double dS2 = (d.heat_cond || d.heat_fric) ? pow(m1 / dens, 2.0 / 3.0) : 0.0;
        if (fr_sta > 0.) {
          double du[3], tg[3];
          for (int k = 0; k < 3; ++k) du[k] = xp[k] - x[k] - v2[k] * dt;
          const double dn = du[0] * n2[0] + du[1] * n2[1] + du[2] * n2[2];
          for (int k = 0; k < 3; ++k) tg[k] = kij * (du[k] - dn * n2[k]);
          const double ntg = sqrt(tg[0] * tg[0] + tg[1] * tg[1] + tg[2] * tg[2]);
          const double ncf = sqrt(cf[0] * cf[0] + cf[1] * cf[1] + cf[2] * cf[2]);
          if (ntg < fr_sta * ncf) {
            for (int k = 0; k < 3; ++k) {
              cf[k] -= tg[k] / m1;
              a[k] -= tg[k] / m1;
            }
          } else {
            double td[3];
            for (int k = 0; k < 3; ++k) {
              td[k] = fr_dyn * ncf * tg[k] / ntg;
              cf[k] -= td[k];
              a[k] -= td[k] / m1;
            }
            if (d.heat_fric) {
              // friction work as heat (Source/Contact_Wang.cpp:291-300)
              const double afv = fabs(td[0] * (v[0] - v2[0]) + td[1] * (v[1] - v2[1]) + td[2] * (v[2] - v2[2]));
              qf = afv * dens / m1;
              cs = sqrt(td[0] * td[0] + td[1] * td[1] + td[2] * td[2]) / dS2;
              fh = afv / dS2;
            }
          }
        }
        cfsum += sqrt(cf[0] * cf[0] + cf[1] * cf[1] + cf[2] * cf[2]);
        for (int m = 0; m < kMaxMesh; ++m)
          if (m == mi)
            for (int k = 0; k < 3; ++k) {
              cfm[m][k] += cf[k];
              cfi[m][k] += cf[k];
            }
        creact += (a[0] * n2[0] + a[1] * n2[1] + a[2] * n2[2]) * m1;
        extw += cf[0] * v2[0] + cf[1] * v2[1] + cf[2] * v2[2];
        // contact conductance, Fraser 3.121 (Source/Contact_Wang.cpp:320-324)
        if (d.heat_cond) qc = dens * d.hc * dS2 * (d.rT[r] - d.T[i]) / m1;
      }
      d.acc[i] = make_double4(a[0], a[1], a[2], a4.w);
    }
    d.cforce[i] = make_double4(cf[0], cf[1], cf[2], 0.0);
    if (d.gcf && cnt > 0)
      for (int m = 0; m < d.nmesh; ++m) d.gcf[(long long)m * d.npad + i] = make_double4(cfi[m][0], cfi[m][1], cfi[m][2], 0.0);
    if (d.qfric) {
      d.qfric[i] = qf;
      d.fhfl[i] = fh;
      d.cshear[i] = cs;
      d.qcont[i] = qc;
    }
  }
  for (int m = 0; m < d.nmesh; ++m)
    for (int k = 0; k < 3; ++k) {
      const double r = block_reduce<0>(cfm[m][k], sh);
      if (threadIdx.x == 0) part(d, P_CFORCE + 3 * m + k, blockIdx.x) = r;
    }
  const double r1 = block_reduce<0>(cfsum, sh);
  const double r2 = block_reduce<0>(creact, sh);
  const double r3 = block_reduce<0>(extw, sh);
  const double r4 = block_reduce<2>(fts, sh);
  if (threadIdx.x == 0) {
    part(d, P_FTS, blockIdx.x) = r4;
    part(d, P_CFSUM, blockIdx.x) = r1;
    part(d, P_CREACT, blockIdx.x) = r2;
    // the work takes the step size of the contact evaluation, before any
    // adaptive update of the step (Source/Contact_Wang.cpp:344)
    part(d, P_EXTW, blockIdx.x) = r3 * dt;
  }
}

// Fraser's (LAW 0, Source/Contact.cpp:223-554), Seo's (LAW 2,
// Source/Contact.cpp:562-770) and LS-Dyna's (LAW 4, Source/Contact_LS.cpp:
// 15-292) contact laws, per particle over its partners in index order.  Under
// Leapfrog none of them adds its force to a: contforce (assigned per pair,
// friction terms added or assigned after it) and the sums are outputs; only
// Fraser's Fr_Bound friction changes a, removing its tangential part.
//   Fraser: pairs approaching (delta_ = -n.v_r > 0) whose time to contact
//     t_c = (h + pplane - n.x) / (-delta_) is below dt, contact point
//     x + v t_c - h n; penetration (dt - t_c) delta_; stiffness
//     PFAC cont_stiff; a sliding pair (|v_t| > 1e-3) assigns
//     contforce = -friction_dyn |contforce| t / m.  The static branch reads
//     a force the reference never sets before it and adds nothing here.
//   Seo: dist = n.x - pplane < h, contact point x - dist n; stiffness
//     PFAC cont_stiff; static friction when |m a_t| < friction_sta
//     |contforce|: contforce -= PFAC cont_stiff (v_r dt)_t / m.
//   LS-Dyna: Wang's geometry (predicted position), stiffness
//     2 m / dt^2 PFAC; friction: the trial force -PFAC m v_r / dt returned
//     to the cone friction_sta |contforce| (the reference's old tangential
//     force is never set: zero) and added; contact_reaction_sum and the
//     external work as Wang's; the contact heat fields are reset.
// dt_fext = 2 m |v| / |contforce| per pair: Domain::min_force_ts takes the
// least positive one (Fraser, Seo) or the least (LS-Dyna) below 1000.
template <int LAW>
WF_KERNEL void k_contact_law(Dev d, int cur, double dt) {
  if (dt < 0) dt = d.flags->dt;
  __shared__ double sh[kBlock / 64];
  const int i = blockIdx.x * kBlock + threadIdx.x;
  double cfsum = 0.0, creact = 0.0, extw = 0.0, fts = INFINITY;
  if (i < d.n) {
    double cf[3] = {0, 0, 0};
    const int cnt = d.ccnt[i];
    if (cnt > 0) {
      const double4 x4 = d.xh[cur][i];
      const double4 v4 = d.vm[i];
      const double4 a4 = d.acc[i];
      const double x[3] = {x4.x, x4.y, x4.z}, v[3] = {v4.x, v4.y, v4.z};
      double a[3] = {a4.x, a4.y, a4.z};
      const double h = x4.w, m1 = v4.w;
      const DevMat &Mi = d.mats[d.mat[i]];
      double fr_sta = Mi.fr_sta >= 0.0 ? Mi.fr_sta : d.fr_sta;
      double fr_dyn = Mi.fr_sta >= 0.0 ? Mi.fr_dyn : d.fr_dyn;
      // friction_function Linear (Source/Contact_LS.cpp:217-220)
      if (LAW == 4 && d.fric_linear) fr_sta = fr_dyn = d.fr_m * d.T[i] + d.fr_b;
      const double ks = (LAW == 0 || LAW == 2) ? d.cstiff[i] : 0.0;
      const double nv = sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
      for (int q = 0; q < cnt; ++q) {
        const int r = d.cidx[(long long)q * d.npad + i];
        const double4 en = d.enorm[r];
        const double n2[3] = {en.x, en.y, en.z};
        const double4 v24 = d.rv[r];
        const double v2[3] = {v24.x, v24.y, v24.z};
        const double vr[3] = {v[0] - v2[0], v[1] - v2[1], v[2] - v2[2]};
        const double delta_ = -(n2[0] * vr[0] + n2[1] * vr[1] + n2[2] * vr[2]);
        double qj[3], delta;
        if (LAW == 0) {
          if (!(delta_ > 0)) continue;
          const double tc = (h + en.w - (n2[0] * x[0] + n2[1] * x[1] + n2[2] * x[2])) / (-delta_);
          if (!(tc < dt)) continue;
          for (int k = 0; k < 3; ++k) qj[k] = x[k] + (v[k] * tc) - (h * n2[k]);
          delta = (dt - tc) * delta_;
        } else {
          double xp[3];
          for (int k = 0; k < 3; ++k) xp[k] = LAW == 4 ? x[k] + v[k] * dt + a[k] * dt * dt / 2.0 : x[k];
          const double dist = (n2[0] * xp[0] + n2[1] * xp[1] + n2[2] * xp[2]) - en.w;
          if (!(dist < h)) continue;
          for (int k = 0; k < 3; ++k) qj[k] = x[k] - dist * n2[k];
          delta = h - dist;
        }
        const int4 el = d.elem[r];
        const int nd[3] = {el.x, el.y, el.z};
        bool inside = true;
        for (int ii = 0; ii < 3 && inside; ++ii) {
          const int jj = ii + 1 > 2 ? 0 : ii + 1;
          const double4 ni = d.node[nd[ii]], nj = d.node[nd[jj]];
          const double ea[3] = {nj.x - ni.x, nj.y - ni.y, nj.z - ni.z};
          const double eb[3] = {qj[0] - ni.x, qj[1] - ni.y, qj[2] - ni.z};
          double c[3];
          cross_d(ea, eb, c);
          if (c[0] * n2[0] + c[1] * n2[1] + c[2] * n2[2] < 0.0) inside = false;
        }
        if (!inside) continue;
        const double kij = LAW == 4 ? 2.0 * m1 / (dt * dt) * d.pfac : d.pfac * ks;
        const double omega = sqrt(kij / m1);
        const double psi = 2. * m1 * omega * d.dfac;
        const double ncf0 = kij * delta - psi * delta_;
        for (int k = 0; k < 3; ++k) cf[k] = ncf0 * n2[k];
        const double nc = sqrt(cf[0] * cf[0] + cf[1] * cf[1] + cf[2] * cf[2]);
        if (LAW != 4) cfsum += nc;
        const double dt_fext = 1. * (m1 * 2. * nv / nc);
        if (dt_fext < 1000. && dt_fext < fts && (LAW == 4 || dt_fext > 0)) fts = dt_fext;
        const double an = a[0] * n2[0] + a[1] * n2[1] + a[2] * n2[2];
        const double atg[3] = {a[0] - an * n2[0], a[1] - an * n2[1], a[2] - an * n2[2]};
        if (LAW == 0) {
          if (d.fric_bound) {
            for (int k = 0; k < 3; ++k) a[k] -= atg[k];
          } else if (fr_dyn > 0.) {
            double tg[3];
            for (int k = 0; k < 3; ++k) tg[k] = vr[k] + delta_ * n2[k];
            const double ntg = sqrt(tg[0] * tg[0] + tg[1] * tg[1] + tg[2] * tg[2]);
            if (ntg > 1.e-3)
              for (int k = 0; k < 3; ++k) cf[k] = -(fr_dyn * nc * (tg[k] / ntg)) / m1;
          }
        } else if (LAW == 2) {
          double du[3], tg[3], rt[3];
          for (int k = 0; k < 3; ++k) du[k] = vr[k] * dt;
          const double dn = du[0] * n2[0] + du[1] * n2[1] + du[2] * n2[2];
          for (int k = 0; k < 3; ++k) tg[k] = kij * (du[k] - dn * n2[k]);
          for (int k = 0; k < 3; ++k) rt[k] = atg[k] * m1;
          if (fr_sta > 0. && sqrt(rt[0] * rt[0] + rt[1] * rt[1] + rt[2] * rt[2]) < fr_sta * nc)
            for (int k = 0; k < 3; ++k) cf[k] -= tg[k] / m1;
        } else {
          if (fr_sta > 0.) {
            double fs[3];
            for (int k = 0; k < 3; ++k) fs[k] = 0.0 - d.pfac * m1 * vr[k] / dt;
            const double fy = fr_sta * nc;
            const double nfs = sqrt(fs[0] * fs[0] + fs[1] * fs[1] + fs[2] * fs[2]);
            for (int k = 0; k < 3; ++k) cf[k] += nfs > fy ? fy * fs[k] / nfs : fs[k];
          }
          cfsum += sqrt(cf[0] * cf[0] + cf[1] * cf[1] + cf[2] * cf[2]);
          creact += an * m1;
          extw += cf[0] * v2[0] + cf[1] * v2[1] + cf[2] * v2[2];
        }
      }
      if (LAW == 0 && d.fric_bound) d.acc[i] = make_double4(a[0], a[1], a[2], a4.w);
    }
    d.cforce[i] = make_double4(cf[0], cf[1], cf[2], 0.0);
    // the laws leave m_contact_force alone: no per-group contact sums
    if (d.gcf && cnt > 0)
      for (int m = 0; m < d.nmesh; ++m) d.gcf[(long long)m * d.npad + i] = make_double4(0.0, 0.0, 0.0, 0.0);
    if (d.qfric) {
      d.qfric[i] = 0.0;
      d.fhfl[i] = 0.0;
      d.cshear[i] = 0.0;
      d.qcont[i] = 0.0;
    }
  }
  const double r1 = block_reduce<0>(cfsum, sh);
  const double r2 = block_reduce<0>(creact, sh);
  const double r3 = block_reduce<0>(extw, sh);
  const double r4 = block_reduce<2>(fts, sh);
  if (threadIdx.x == 0) {
    for (int m = 0; m < d.nmesh; ++m)
      for (int k = 0; k < 3; ++k) part(d, P_CFORCE + 3 * m + k, blockIdx.x) = 0.0;
    part(d, P_FTS, blockIdx.x) = r4;
    part(d, P_CFSUM, blockIdx.x) = r1;
    part(d, P_CREACT, blockIdx.x) = r2;
    part(d, P_EXTW, blockIdx.x) = r3 * dt;
  }
}

// Domain::CalcForce2233 (Source/Interaction.cpp:25-333) as
// LastComputeAcceleration applies it to every pair (Source/Domain.cpp:
// 1700-1709), as one FP64 gather per particle over its row: the pair's
// terms for particle i are the reference's for P1 with (P1, P2) = (i, j)
// (each term is odd or even under the swap, so the second particle's terms
// are the same formula from its side).  Per neighbour: a += m_j g.(sigma_i/
// rho_i^2 + sigma_j/rho_j^2 + Pi), dDensity from (m_j/rho_j) v_ij.g (times
// rho_i), StrainRate / RotationRate with the float weight (float)(m_j/rho_j)
// (`float mj_dj`, Source/Interaction.cpp:262), ZWab += (float)(m_j/rho_j) W,
// VXSPH += XSPH m_j / ((rho_i + rho_j)/2) W (v_j - v_i) and, when shepard,
// SumDen += m_j W; g = GK x_ij or (GK L_i) x_ij under the gradient
// correction.  GradientType 0, free-free pairs, no tensile instability.
template <bool GC>
__global__ __launch_bounds__(kBlock) void k_force2233(Dev d, int cur, double xsph, int shepard) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= d.n) return;
  using S = Src<false>;
  const long long np = d.npad;
  double a[3] = {0, 0, 0}, s = 0, sr[6] = {0, 0, 0, 0, 0, 0}, w[3] = {0, 0, 0}, zw = 0, sd = 0;
  double vx[3] = {0, 0, 0};
  const double rhoi = d.rho[cur][i];
  if (d.group[i] >= 0) {
    double Li[6];
    own_corr<GC>(d, i, Li);
    const DevMat &M = d.mats[d.mat[i]];
    const double alpha = M.alpha, beta = M.beta, cs = M.Cs;
    const bool av = (alpha != 0.0 || beta != 0.0);
    const double4 xi = S::x(d, cur, i), vi = S::v(d, i);
    double ti[6], rho_i;
    S::srec(d, i, ti, rho_i);
    const KH<double> ki = kern_h_t<double>(xi.w, d.dim);
    const HbmJ<false> g{d, cur, i};
    for_each_nb(g, d.nnb[i], 0, 1, [&](int j) {
      const double4 xj = g.x(j), vj = g.v(j);
      double tj[6], rho_j;
      g.srec(j, tj, rho_j);
      const KH<double> kh = S::kh(ki, xi, xj);
      const double dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
      const double r2 = dx * dx + dy * dy + dz * dz;
      const double GK = gk_t<double>(r2, kh);
      const double q = r2 > 0.0 ? sqrt(r2) * kh.ih : 0.0;
      // W's constant C (Source/Functions.cpp:32): 1/(pi h^3), 10/(7 pi h^2) in 2D
      const double K = w_shape<double>(q) * (d.dim == 2 ? kh.ih * kh.ih * (10.0 / (7.0 * M_PI))
                                                        : kh.ih * kh.ih * kh.ih * (1.0 / M_PI));
      const double vdx = vi.x - vj.x, vdy = vi.y - vj.y, vdz = vi.z - vj.z;
      const double vdot = vdx * dx + vdy * dy + vdz * dz;
      double pi = 0.0;
      if (av && vdot < 0.0) {
        const double mu = kh.h * vdot / (r2 + 0.01 * kh.h * kh.h);
        pi = (alpha * cs * mu + beta * mu * mu) / (0.5 * (rho_i + rho_j));
      }
      double ex, ey, ez;
      corr_dir<GC>(Li, dx, dy, dz, ex, ey, ez);
      const double gx = GK * ex, gy = GK * ey, gz = GK * ez;
      const double Mxx = ti[XX] + tj[XX] + pi, Myy = ti[YY] + tj[YY] + pi, Mzz = ti[ZZ] + tj[ZZ] + pi;
      const double Mxy = ti[XY] + tj[XY], Mxz = ti[XZ] + tj[XZ], Myz = ti[YZ] + tj[YZ];
      const double mj = vj.w;
      a[0] += mj * (gx * Mxx + gy * Mxy + gz * Mxz);
      a[1] += mj * (gx * Mxy + gy * Myy + gz * Myz);
      a[2] += mj * (gx * Mxz + gy * Myz + gz * Mzz);
      const double volj = S::vol(d, cur, j, xj);
      s += volj * (vdx * gx + vdy * gy + vdz * gz);
      const double fw = (double)(float)volj;
      const double c = fw * (-0.5 * GK);
      sr[XX] += c * (2.0 * vdx * ex);
      sr[YY] += c * (2.0 * vdy * ey);
      sr[ZZ] += c * (2.0 * vdz * ez);
      sr[XY] += c * (vdx * ey + vdy * ex);
      sr[XZ] += c * (vdx * ez + vdz * ex);
      sr[YZ] += c * (vdy * ez + vdz * ey);
      w[0] += c * (vdx * ey - vdy * ex);
      w[1] += c * (vdx * ez - vdz * ex);
      w[2] += c * (vdy * ez - vdz * ey);
      // rows are padded with the particle itself: its pair terms above are
      // exact zeros, the kernel sums must skip it
      const bool real = j != i;
      zw += real ? fw * K : 0.0;
      const double xf = xsph * mj / (0.5 * (rhoi + d.rho[cur][j])) * K;
      vx[0] += xf * -vdx;
      vx[1] += xf * -vdy;
      vx[2] += xf * -vdz;
      if (shepard && real) sd += mj * K;
    });
  }
  if (d.dim == 2 && !GC) a[2] = 0.0;  // plane strain (Source/Interaction.cpp:237)
  const double4 a4 = d.acc[i];
  d.acc[i] = make_double4(a[0], a[1], a[2], a4.w);
  d.drho[i] = s * rhoi;
  for (int k = 0; k < 6; ++k) d.sr[k * np + i] = sr[k];
  for (int k = 0; k < 3; ++k) d.rr[k * np + i] = w[k];
  d.zwab[i] = zw;
  d.vxsph[i] = make_double4(vx[0], vx[1], vx[2], 0.0);
  d.sumden[i] = sd;
}

void launch_force2233(const Dev &d, hipStream_t st, int cur, double xsph, int shepard) {
  if (d.gc_on)
    k_force2233<true><<<d.nblocks, kBlock, 0, st>>>(d, cur, xsph, shepard);
  else
    k_force2233<false><<<d.nblocks, kBlock, 0, st>>>(d, cur, xsph, shepard);
}

// Per-group sums (wf_set_group_sums).  what 0: the reaction of zone gzone,
// sum of m a over the group's particles carrying that id, read where the
// zone reactions are (after the acceleration pass, before contact and the
// BCs); what 1: the contact force each rigid mesh exerts on the group (after
// contact).  A block sums one chunk of at most kGroupChunk particles (thread
// t takes every kGroupThreads-th, all of a thread's loads in flight); the
// block of a group that finishes last (a ticket counter, reset by it) adds
// the group's chunk sums in chunk order, so the sums are deterministic.
//
// The pass reads 8 bytes per particle and is bound by the latency of its two
// dependent loads.  One block per group walking all of it left 64 blocks on
// the chip: 183 us per step for 64 groups of 9.4 thousand particles and two
// meshes; with chunks 18 us (30 us with a fence before the ticket).
constexpr int kGroupThreads = 256;
constexpr int kGroupPer = kGroupChunk / kGroupThreads;
__global__ __launch_bounds__(kGroupThreads) void k_group_sums(Dev d, int what) {
  __shared__ double sh[kGroupThreads / 64][3 * kMaxMesh];
  __shared__ int last;
  const int4 ch = d.gchunk[blockIdx.x];
  const int g = ch.x, nm = what == 0 ? 1 : d.nmesh, tid = threadIdx.x;
  int idx[kGroupPer];
  bool on[kGroupPer], any = false;
#pragma unroll
  for (int u = 0; u < kGroupPer; ++u) {
    const int p = ch.y + u * kGroupThreads + tid;
    on[u] = p < ch.z;
    idx[u] = on[u] ? d.gidx[p] : 0;
  }
#pragma unroll
  for (int u = 0; u < kGroupPer; ++u) {
    on[u] = on[u] && (what == 0 ? d.id[idx[u]] == d.gzone : d.ccnt[idx[u]] > 0);
    any = any || on[u];
  }
  // (most chunks hold no particle of the zone or in contact)
  if (__syncthreads_or(any)) {
    for (int m = 0; m < nm; ++m) {
      double s[3] = {0, 0, 0};
#pragma unroll
      for (int u = 0; u < kGroupPer; ++u) {
        if (!on[u]) continue;
        if (what == 0) {
          const double4 a = d.acc[idx[u]];
          const double w = d.vm[idx[u]].w;
          s[0] += w * a.x, s[1] += w * a.y, s[2] += w * a.z;
        } else {
          const double4 f = d.gcf[(long long)m * d.npad + idx[u]];
          s[0] += f.x, s[1] += f.y, s[2] += f.z;
        }
      }
      for (int k = 0; k < 3; ++k) {
        const double r = wave_sum(s[k]);
        if ((tid & 63) == 0) sh[tid >> 6][3 * m + k] = r;
      }
    }
  } else if (tid < 3 * nm) {
    for (int w = 0; w < kGroupThreads / 64; ++w) sh[w][tid] = 0.0;
  }
  __syncthreads();
  const int nch = d.gnch[g];
  if (tid < 3 * nm) {
    double r = sh[0][tid];
    for (int w = 1; w < kGroupThreads / 64; ++w) r += sh[w][tid];
    put_agent(&d.gpart[(long long)blockIdx.x * kMaxMesh * 3 + tid], r);
  }
  stores_done();
  __syncthreads();
  if (tid == 0) last = atomicAdd(&d.gticket[g], 1) == nch - 1;
  __syncthreads();
  if (!last) return;
  if (tid < 3 * nm) {
    double r = 0.0;
#pragma unroll 8
    for (int c = 0; c < nch; ++c)
      r += get_agent(&d.gpart[(long long)(ch.w + c) * kMaxMesh * 3 + tid]);
    const long long slot = (d.flags->step % d.ghist_cap) * d.ngroups + g;
    if (what == 0) d.gr_hist[slot * 3 + tid] = r;
    else d.gc_hist[slot * kMaxMesh * 3 + tid] = r;
  }
  if (tid == 0) d.gticket[g] = 0;
}

void launch_group_sums(const Dev &d, hipStream_t st, int what) {
  if (d.ngroups > 0) k_group_sums<<<d.ngchunks, kGroupThreads, 0, st>>>(d, what);
}

// the drift of the rigid particles alone, for a step run in parts (a whole
// step drifts them with the mesh update)
WF_KERNEL void k_rigid_drift(Dev d, double dt) {
  if (dt < 0) dt = d.flags->dt;
  const int r = blockIdx.x * kBlock + threadIdx.x;
  if (r >= d.nrig) return;
  double4 x = d.rx[r];
  const double4 v = d.rv[r];
  x.x += v.x * dt;
  x.y += v.y * dt;
  x.z += v.z * dt;
  d.rx[r] = x;
}

// Blocks of 16 particles spread the partner search of small models over the
// chip, but cost 2 us on steps without a search once there are a thousand of
// them.  They are taken up to 32768 particles where the rigid surface is fine
// against the model (a rigid particle or more for 16 of the model's), so that
// its particles have many candidates.  Us per step with a search every 5, blocks
// of 16 against 128 particles, rigid surfaces of 256, 576, 1024, 2304 and, at
// 18k and 30k, 8192 particles:
//   1.3k  14 15   19 20   25 28   43 51
//   9k    14.3 13.9   14.6 15.2   16 17   21 21
//   18k   15.2 13.7   15.8 15.1   15.5 16.2   19.5 20.6   19 75
//   30k   16.1 13.7   16.7 14.6   16.7 15.2   18.3 18.7   48 65
constexpr int kSurfSmall = 32768, kSurfFine = 16;
void launch_surface(const Dev &d, hipStream_t st, int cur, int setup) {
  if (setup == 0 && d.n <= kSurfSmall && d.n <= kSurfFine * (long long)d.nrig)
    k_surface<16><<<(d.n + 15) / 16, kBlock, 0, st>>>(d, cur, setup);
  else k_surface<kBlock><<<nblk(d.n), kBlock, 0, st>>>(d, cur, setup);
}
void launch_rigid_bc(const Dev &d, hipStream_t st, const BcTable &bc) {
  k_rigid_bc<<<nblk(d.nrig), kBlock, 0, st>>>(d, bc);
}
void launch_contact(const Dev &d, hipStream_t st, int cur, double dt, int law) {
  switch (law) {
    case 0: k_contact_law<0><<<d.nblocks, kBlock, 0, st>>>(d, cur, dt); break;
    case 2: k_contact_law<2><<<d.nblocks, kBlock, 0, st>>>(d, cur, dt); break;
    case 4: k_contact_law<4><<<d.nblocks, kBlock, 0, st>>>(d, cur, dt); break;
    default: k_contact<<<d.nblocks, kBlock, 0, st>>>(d, cur, dt);
  }
}
void launch_rigid_drift(const Dev &d, hipStream_t st, double dt) {
  k_rigid_drift<<<(d.nrig + kBlock - 1) / kBlock, kBlock, 0, st>>>(d, dt);
}

// ---------------------------------------------------------------------------
// utilities

WF_KERNEL void k_max_pl(Dev d) {
  __shared__ double sh[kBlock / 64];
  const int i = blockIdx.x * kBlock + threadIdx.x;
  const double v = i < d.n ? d.pl[i] : 0.0;
  const double r = block_reduce<1>(v, sh);
  if (threadIdx.x == 0) part(d, P_MAXT, blockIdx.x) = r;
}

__global__ __launch_bounds__(256) void k_max_pl_final(Dev d) {
  __shared__ double sh[16];
  double v = 0.0;
  for (int b = threadIdx.x; b < d.nblocks; b += blockDim.x) v = fmax(v, part(d, P_MAXT, b));
  const double r = block_reduce<1>(v, sh);
  if (threadIdx.x == 0) d.scalars[S_MAXPL] = r;
}

// rebuild every FP32 shadow from the FP64 state (set-up and host writes)
WF_KERNEL void k_shadows(Dev d, int cur) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= d.n) return;
  const double *o = d.mats[d.mat[i]].xc;
  for (int b = 0; b < 2; ++b) {
    const double4 x = d.xh[b][i];
    d.xhf[b][i] = make_float4((float)(x.x - o[0]), (float)(x.y - o[1]), (float)(x.z - o[2]), (float)d.vol[b][i]);
  }
  const double4 v = d.vm[i];
  d.vmf[i] = make_float4((float)v.x, (float)v.y, (float)v.z, (float)v.w);
  const StressRec r = d.srec[i];
  StressRecF f;
  for (int k = 0; k < 6; ++k) f.t[k] = (float)(r.s[k] * r.irho2);
  f.rho = (float)r.rho;
  f.pad = 0.0f;
  d.srecf[i] = f;
  const DevMat &M = d.mats[d.mat[i]];
  const double rho = d.rho[cur][i];
  d.prf[i] = (float)((M.P0 + M.Cs * M.Cs * (rho - M.ref_density)) / (rho * rho));
}

void launch_shadows(const Dev &d, hipStream_t st, int cur) {
  if (d.mixed) k_shadows<<<nblk(d.n), kBlock, 0, st>>>(d, cur);
}

void launch_max_pl(const Dev &d, hipStream_t st) {
  k_max_pl<<<d.nblocks, kBlock, 0, st>>>(d);
  k_max_pl_final<<<1, 256, 0, st>>>(d);
}

}  // namespace wf
