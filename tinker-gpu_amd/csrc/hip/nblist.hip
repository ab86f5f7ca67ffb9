// Spatial neighbor list for gfx950.
//
// Replaces the reference's 32-atom Hilbert block list (src/cu/spatial.cu:101-960,
// include/ff/spatial.h) with a wave64 design:
//  1. atoms are binned into cells of edge >= (cutoff + buffer)/2 and sorted
//     by (Morton code of the cell, original index) — a counting sort whose
//     within-cell order is then fixed by ranking each cell's atoms, so the
//     order is deterministic;
//  2. every atom gets its own full neighbor list (both directions) of atoms
//     within cutoff + buffer: 64 consecutive atoms share one walk over the
//     cells within two of theirs, kept to what is near their bounding box;
//  3. lists are stored per wavefront of 64 consecutive sorted atoms,
//     k-major, padded to the longest list of the wave.
// Each entry packs the neighbor's sorted index and its scale class (the
// reference's exclusion bit masks, spatial.h si1..si4).  Pair kernels walk
// their own atom's list and write only their own atom's sums: no atomics,
// fixed summation order, bit-reproducible results.
#include <climits>
#include <cstdlib>
#include <cstring>

#include "ctx.hpp"

namespace t9 {
namespace {

constexpr int kScanBlock = 1024;

__device__ __forceinline__ uint32_t spread_bits(uint32_t v) {
  v &= 0x3ff;
  v = (v | (v << 16)) & 0x030000FF;
  v = (v | (v << 8)) & 0x0300F00F;
  v = (v | (v << 4)) & 0x030C30C3;
  v = (v | (v << 2)) & 0x09249249;
  return v;
}

__device__ __forceinline__ int morton3(int x, int y, int z) {
  return (int)(spread_bits(x) | (spread_bits(y) << 1) | (spread_bits(z) << 2));
}

__global__ void k_cell_assign(int n, const double* __restrict__ xyz, double lx, double ly, double lz, int ncx,
                              int ncy, int ncz, int* __restrict__ key, int* __restrict__ rank,
                              int* __restrict__ count, int* __restrict__ cellc_orig) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double fx = xyz[3 * i] / lx, fy = xyz[3 * i + 1] / ly, fz = xyz[3 * i + 2] / lz;
  fx -= floor(fx);
  fy -= floor(fy);
  fz -= floor(fz);
  const int cx = min(ncx - 1, (int)(fx * ncx));
  const int cy = min(ncy - 1, (int)(fy * ncy));
  const int cz = min(ncz - 1, (int)(fz * ncz));
  const int k = morton3(cx, cy, cz);
  key[i] = k;
  cellc_orig[i] = cx | (cy << 10) | (cz << 20);
  rank[i] = atomicAdd(&count[k], 1);
}

// Exclusive scan of m values into out[0..m-1] by one workgroup, and the sum
// into out[m]; every thread returns the sum.  Each thread sums a contiguous
// segment, the segment sums are scanned across the wavefront by shuffles and
// across the wavefronts through LDS (one barrier).
__device__ __forceinline__ long long block_scan(const long long* __restrict__ in, long long* __restrict__ out, int m) {
  __shared__ long long wsum[kScanBlock / 64];
  const int per = (m + kScanBlock - 1) / kScanBlock;
  const int b = min(m, (int)threadIdx.x * per), e = min(m, b + per);
  long long sum = 0;
  for (int t0 = b; t0 < e; t0 += 8) {  // 8 loads in flight
    long long v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = t0 + u < e ? in[t0 + u] : 0;
#pragma unroll
    for (int u = 0; u < 8; ++u) sum += v[u];
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  long long incl = sum;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const long long y = __shfl_up(incl, o, 64);
    if (lane >= o) incl += y;
  }
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  long long run = incl - sum, all = 0;
  for (int u = 0; u < kScanBlock / 64; ++u) {
    run += u < w ? wsum[u] : 0;
    all += wsum[u];
  }
  for (int t0 = b; t0 < e; t0 += 8) {
    long long v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = t0 + u < e ? in[t0 + u] : 0;
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (t0 + u < e) {
        out[t0 + u] = run;
        run += v[u];
      }
  }
  if (threadIdx.x == 0) out[m] = all;
  return all;
}

// One workgroup each: the largest group count of the waves into tot[0], and
// per list the offsets of the waves' slabs and their total into tot[1 + list]
// (one launch and one readback instead of three each).
__global__ __launch_bounds__(kScanBlock) void k_list_totals(int nw, const int* __restrict__ ngroup,
                                                            const long long* __restrict__ sm,
                                                            long long* __restrict__ off_m,
                                                            const long long* __restrict__ sv,
                                                            long long* __restrict__ off_v,
                                                            long long* __restrict__ tot) {
  if (blockIdx.x > 0) {
    const long long all = blockIdx.x == 1 ? block_scan(sm, off_m, nw) : block_scan(sv, off_v, nw);
    if (threadIdx.x == 0) tot[blockIdx.x] = all;
    return;
  }
  __shared__ int top[kScanBlock / 64];
  int v = 0;
  for (int w = threadIdx.x; w < nw; w += kScanBlock) v = max(v, ngroup[w]);
  for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
  if ((threadIdx.x & 63) == 0) top[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int u = 0; u < kScanBlock / 64; ++u) v = max(v, top[u]);
    tot[0] = v;
    if (!sv) tot[2] = 0;
  }
}

__global__ void k_cell_scatter(int n, const int* __restrict__ key, const int* __restrict__ rank,
                               const int* __restrict__ start, int* __restrict__ unsorted) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) unsorted[start[key[i]] + rank[i]] = i;
}

// Order each cell's atoms by original index: one wavefront per cell, an
// atom's place is the number of the cell's atoms below it (a thread per cell
// sorting in memory took 67 us for 32,768 keys, 17 atoms per cell).
__global__ __launch_bounds__(256) void k_cell_sort(int nkeys, const int* __restrict__ start,
                                                   const int* __restrict__ count, const int* __restrict__ unsorted,
                                                   int* __restrict__ perm) {
  const int k = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (k >= nkeys) return;
  const int s0 = start[k], c = count[k];
  for (int a0 = 0; a0 < c; a0 += 64) {
    const int v = a0 + lane < c ? unsorted[s0 + a0 + lane] : 0x7fffffff;
    int rank = 0;
    for (int b0 = 0; b0 < c; b0 += 64) {
      const int u = b0 + lane < c ? unsorted[s0 + b0 + lane] : 0x7fffffff;
      const int m = min(64, c - b0);
      for (int t = 0; t < m; ++t) rank += __builtin_amdgcn_readlane(u, t) < v ? 1 : 0;
    }
    if (a0 + lane < c) perm[s0 + rank] = v;
  }
}

// Exclusive scan of the cell counts in two launches over chunks of 1024: the
// chunk totals, then each chunk adds the totals before it.
__global__ __launch_bounds__(kScanBlock) void k_count_sums(const int* __restrict__ in, int* __restrict__ csum, int m) {
  __shared__ int ws[kScanBlock / 64];
  const int t = blockIdx.x * kScanBlock + threadIdx.x;
  int v = t < m ? in[t] : 0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    int a = 0;
    for (int u = 0; u < kScanBlock / 64; ++u) a += ws[u];
    csum[blockIdx.x] = a;
  }
}
__global__ __launch_bounds__(kScanBlock) void k_count_scan(const int* __restrict__ in, const int* __restrict__ csum,
                                                           int* __restrict__ out, int m) {
  __shared__ int ws[kScanBlock / 64], wc[kScanBlock / 64];
  const int t = blockIdx.x * kScanBlock + threadIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int before = 0;
  for (int b = threadIdx.x; b < (int)blockIdx.x; b += kScanBlock) before += csum[b];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o, 64);
  const int c = t < m ? in[t] : 0;
  int incl = c;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(incl, o, 64);
    if (lane >= o) incl += y;
  }
  if (lane == 63) ws[w] = incl;
  if (lane == 0) wc[w] = before;
  __syncthreads();
  int run = incl - c;
  for (int u = 0; u < kScanBlock / 64; ++u) run += wc[u] + (u < w ? ws[u] : 0);
  if (t < m) out[t] = run;
}

__global__ void k_identity(int n, int* __restrict__ perm) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) perm[i] = i;
}

template <class real>
__global__ void k_build_sorted(int n, const int* __restrict__ perm, int* __restrict__ iperm,
                               const double* __restrict__ xyz, double* __restrict__ xyz_last, double3 vorg,
                               double3 vlen, int periodic, PosRec<real>* __restrict__ pos,
                               const int* __restrict__ cellc_orig, int* __restrict__ cellc,
                               const double* __restrict__ polarity_o, const double* __restrict__ pdamp_o,
                               const int* __restrict__ jpolar_o, real* __restrict__ polarity,
                               real* __restrict__ polinv, real* __restrict__ pdamp, int* __restrict__ jpolar) {
  int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  int i = perm[s];
  iperm[i] = s;
  double x = xyz[3 * i], y = xyz[3 * i + 1], z = xyz[3 * i + 2];
  xyz_last[3 * i] = x;
  xyz_last[3 * i + 1] = y;
  xyz_last[3 * i + 2] = z;
  const double org[3] = {vorg.x, vorg.y, vorg.z}, len[3] = {vlen.x, vlen.y, vlen.z};
  pos[s] = make_pos<real>(x, y, z, pdamp_o[i] > 0 ? 1.0 / pdamp_o[i] : 0.0, org, len, periodic);
  if (cellc_orig) cellc[s] = cellc_orig[i];
  double a = polarity_o[i];
  polarity[s] = (real)a;
  polinv[s] = (real)(1.0 / (a > 1e-16 ? a : 1e-16));
  pdamp[s] = (real)pdamp_o[i];
  jpolar[s] = jpolar_o[i];
}

template <class real>
__global__ void k_refresh_pos(int n, const int* __restrict__ perm, const double* __restrict__ xyz, double3 vorg,
                              double3 vlen, int periodic, const double* __restrict__ pdamp_o,
                              PosRec<real>* __restrict__ pos) {
  int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  int i = perm[s];
  const double org[3] = {vorg.x, vorg.y, vorg.z}, len[3] = {vlen.x, vlen.y, vlen.z};
  pos[s] = make_pos<real>(xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2], pdamp_o[i] > 0 ? 1.0 / pdamp_o[i] : 0.0, org,
                          len, periodic);
}

// The two lists share one scan over the candidate cells: the multipole list
// (atoms within rm) and the vdW list (sites within rv, sites read from vpos).
//
// A build is two kernels.  k_nb_masks finds the candidates and tests them: a
// workgroup of 8 or 16 wavefronts takes 64 consecutive atoms; its wavefronts
// walk their shares of the surrounding cells, keep what comes within a list's
// radius of the bounding box of the 64 atoms (or of their vdW sites), and the
// kept candidates of all of them are tested in dense groups of 64 (lane = candidate when it is loaded, lane
// = atom while the group is read back candidate by candidate from LDS, one
// broadcast read per record instead of a readlane per word).  The outcome
// is a 64-bit mask per atom, group and list, and the counts.  k_nb_fill turns
// the masks of a list into its entries at the counted offsets.  Testing and
// writing in one kernel spent more than half its time on stores (one per
// candidate and list, each a scattered row) and on the exclusion classes of
// every tested pair: 1,555 us for 96,000 atoms and 193 us per list to pack,
// against 362 and 243 for both lists.
template <class real>
struct ListArgs {
  int n, brute, periodic;
  const PosRec<real>* pos;
  const PosRec<real>* vpos;  // null: no vdW list
  const int* cellc;
  int nc[3];
  const int* cell_start;
  const int* cell_count;
  BoxT<real> box;
  real rm2, rv2;
  real rs2[2], sy, sz;       // the same radii squared in the units of near_test, and its axis ratios
  double reach;              // reach of the candidate search (A)
  double csize[3];           // cell edge (A)
  double flen[3];            // box edge (FP64 positions are wrapped coordinates)
  int *nm, *nv;              // [n] counts
  int *mm, *mv;              // [waves] largest counts
  long long *sm, *sv;        // [waves] slab sizes
  int wave0;                 // first wave of this launch
  int ngmax;                 // groups per wave that the masks hold
  int* ngroup;               // [waves] groups found (above ngmax: not stored)
  int* cand;                 // [waves of the launch][ngmax][64] candidate of each mask bit
  ulonglong2* mask;          // [waves of the launch][ngmax][64] (multipole, vdW) bits per atom
};

constexpr int kParts = 16;  // wavefronts that write a wave of atoms' rows

__device__ __forceinline__ double frac_of(const PosRec<float>& p, int d, const double*) {
  const unsigned v = d == 0 ? (unsigned)p.x : (d == 1 ? (unsigned)p.y : (unsigned)p.z);
  return (double)v * (1.0 / 4294967296.0);
}
__device__ __forceinline__ double frac_of(const PosRec<double>& p, int d, const double* flen) {
  return (d == 0 ? p.x : (d == 1 ? p.y : p.z)) / flen[d];
}

// A lane's scaled partners, as sorted indices: the first 8 in registers, the
// rest read when needed (none for water and most of a protein's atoms).  np:
// the largest count of the wavefront (2 for water), so few are compared.
struct Partners {
  int j[8], code[8];
  int e0, e1, np;
  const int *ej, *ec, *iperm;
  __device__ __forceinline__ void load(int a, int b, const int* __restrict__ ej_, const int* __restrict__ ec_,
                                       const int* __restrict__ iperm_) {
    e0 = a;
    e1 = b;
    ej = ej_;
    ec = ec_;
    iperm = iperm_;
    np = wave_max(b - a);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const bool in = a + k < b;
      j[k] = in ? iperm[ej[a + k]] : -1;
      code[k] = in ? ec[a + k] : 0;
    }
  }
  __device__ __forceinline__ int find(int s) const {
    int c = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      if (k >= np) break;
      c = j[k] == s ? code[k] : c;
    }
    for (int e = e0 + 8; e < e1; ++e)
      if (iperm[ej[e]] == s) c = ec[e];
    return c;
  }
};

__device__ __forceinline__ int wave_min(int v) {
  for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
  return __builtin_amdgcn_readfirstlane(v);
}
// (results in scalar registers: the candidate scan keeps them throughout)
__device__ __forceinline__ double wave_uniform(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readfirstlane((int)(b & 0xffffffffLL));
  const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ float wave_uniform(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}
__device__ __forceinline__ double wave_minf(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
  return wave_uniform(v);
}
__device__ __forceinline__ double wave_maxf(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return wave_uniform(v);
}

__device__ __forceinline__ int wrapc(int x, int nc) {
  x += x < 0 ? nc : 0;
  return x - (x >= nc ? nc : 0);
}

// Wave-uniform broadcast of lane t's value (t uniform).
__device__ __forceinline__ int bcast(int v, int t) { return __builtin_amdgcn_readlane(v, t); }
__device__ __forceinline__ float bcast(float v, int t) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), t));
}
__device__ __forceinline__ double bcast(double v, int t) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), t);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), t);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
template <class real>
__device__ __forceinline__ PosRec<real> bcast(const PosRec<real>& p, int t) {
  PosRec<real> q;
  q.x = bcast(p.x, t);
  q.y = bcast(p.y, t);
  q.z = bcast(p.z, t);
  q.w = bcast(p.w, t);
  return q;
}

// Extent of a wavefront's atoms around a reference atom: the bounding box of
// their minimum-image displacements from it, as centre and half edges.
template <class real>
struct WaveBox {
  PosRec<real> ref;
  real mid[3], half[3];
  // of the lanes with `mine`, around lane `lead` (one of them)
  __device__ __forceinline__ void set(const PosRec<real>& p, const BoxT<real>& box, int lead, bool mine) {
    ref = bcast(p, lead);
    real d[3];
    pair_disp(ref, p, box, d[0], d[1], d[2]);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const double v = mine ? (double)d[q] : 0.0;
      const double lo = wave_minf(v), hi = wave_maxf(v);
      mid[q] = wave_uniform((real)(0.5 * (lo + hi)));
      half[q] = wave_uniform((real)(0.5 * (hi - lo) + 1e-3));  // covers the rounding of the test
    }
  }
  // squared distance of a candidate to the box, under the minimum image
  __device__ __forceinline__ real dist2(const PosRec<real>& p, const BoxT<real>& box, int periodic) const {
    real d[3], s = 0;
    pair_disp(ref, p, box, d[0], d[1], d[2]);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      real t = d[q] - mid[q];
      if (periodic) t -= box.l[q] * t9_rint(t * box.il[q]);
      const real g = fmax((real)0, (t < 0 ? -t : t) - half[q]);
      s += g * g;
    }
    return s;
  }
};

// Negative if b lies within a list's radius of a (rs2: its square in the units
// of the test).  FP32: the fixed-point differences, squared in units of the x
// quantum; the squared radius is a millionth larger than asked, which covers
// the rounding.
__device__ __forceinline__ float near_test(const PosRec<float>& a, const PosRec<float>& b, const ListArgs<float>& A,
                                           float rs2) {
  const float x = (float)(int)((unsigned)b.x - (unsigned)a.x);
  const float y = (float)(int)((unsigned)b.y - (unsigned)a.y);
  const float z = (float)(int)((unsigned)b.z - (unsigned)a.z);
  return fmaf(z * z, A.sz, fmaf(y * y, A.sy, fmaf(x, x, -rs2)));
}
__device__ __forceinline__ double near_test(const PosRec<double>& a, const PosRec<double>& b,
                                            const ListArgs<double>& A, double rs2) {
  double x, y, z;
  pair_disp(a, b, A.box, x, y, z);
  return x * x + y * y + z * z - rs2;
}
// the sign bit of v shifted into m from below
__device__ __forceinline__ unsigned shift_in(unsigned m, float v) {
  return __builtin_amdgcn_alignbit(m, (unsigned)__float_as_int(v), 31);
}
__device__ __forceinline__ unsigned shift_in(unsigned m, double v) {
  return __builtin_amdgcn_alignbit(m, (unsigned)(__double_as_longlong(v) >> 32), 31);
}
// The 64 outcomes of atom a against a group of records, bit t for record t.
template <class real>
__device__ __forceinline__ unsigned long long near_bits(const PosRec<real>& a, const PosRec<real>* g,
                                                        const ListArgs<real>& A, real rs2) {
  unsigned b[2] = {0, 0};
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll 8
    for (int t = 31; t >= 0; --t) b[h] = shift_in(b[h], near_test(a, g[32 * h + t], A, rs2));
  return ((unsigned long long)b[1] << 32) | b[0];
}

// What bounds the scan is the instructions of these tests (12 per pair and
// list in FP32).  So a candidate within reach for the longer list only is kept
// apart, and its group tested for that list alone; and the cells' atoms are
// taken 64 at a time whatever the cells hold (17 each at 96,000 atoms).  593
// -> 362 us there, with the 12 instructions instead of 18.
constexpr int kSeg = 256;  // candidates a wavefront keeps before a batch is tested

// Candidates and masks (see above).  One walk takes a cluster of the atoms:
// all of them when they span at most 4 cells per axis (the usual case: 64
// consecutive atoms in cell Morton order), else, where that order jumps, those
// within one cell of the first atom that is left, and so on.  It visits the
// cells within two of the cluster's, each once (an axis with no more cells
// than that is visited whole), and keeps what lies within reach of the
// cluster's bounding box.  Without cells, one walk over all atoms.  (One walk
// per home cell, without the box, made the workgroups at the jumps and those
// of every box of few cells several times longer than the others: 901 -> 593
// us for 96,000 atoms; the dipoles of 3,000 with their lists 1,462 -> 1,044.)
// The wavefronts take the cells (or the atom range) in P fixed parts, so
// the candidates' order does not depend on scheduling.
template <class real, int P>
__global__ __launch_bounds__(64 * P, 4) void k_nb_masks(ListArgs<real> A) {
  __shared__ int seg[P][kSeg];
  __shared__ int segn[2][P];  // kept from the front and from the back
  __shared__ int more;
  __shared__ int csum[2][P][64];
  __shared__ PosRec<real> grp[P][64], vgrp[P][64];  // the group a wavefront tests
  const int lane = threadIdx.x & 63, part = threadIdx.x >> 6;
  const int lb = xcd_block(), blk = A.wave0 + lb;
  const int s0 = blk * 64 + lane;
  const bool active = s0 < A.n;
  const int s = active ? s0 : A.n - 1;  // idle lanes mirror the last atom
  const auto pi = A.pos[s];
  const bool has_v = A.vpos != nullptr;
  PosRec<real> vi = pi;
  if (has_v) vi = A.vpos[s];
  const int c = A.brute ? 0 : A.cellc[s];
  const int cq[3] = {c & 1023, (c >> 10) & 1023, (c >> 20) & 1023};
  const double reach2 = A.reach * A.reach;
  const bool v_longer = has_v && A.rv2 > A.rm2;
  int cm = 0, cv = 0, gbase = 0;
  unsigned long long todo = __ballot(1);
  while (todo) {
    // the walk's atoms (`mine`); its cells: base r0, size rs; its extent in
    // cells from the leading atom's cell: bl..bh
    const int lead = __builtin_ctzll(todo);
    const bool left_over = (todo >> lane) & 1;
    int h0[3] = {0, 0, 0}, r0[3] = {0, 0, 0}, rs[3] = {1, 1, 1};
    double bl[3] = {0, 0, 0}, bh[3] = {0, 0, 0};
    bool mine = left_over;
    if (!A.brute) {
      int d[3], lo[3], hi[3];
      bool all = true, one = left_over;
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        h0[q] = __builtin_amdgcn_readlane(cq[q], lead);
        d[q] = cq[q] - h0[q];
        d[q] -= 2 * d[q] >= A.nc[q] ? A.nc[q] : 0;
        d[q] += 2 * d[q] < -A.nc[q] ? A.nc[q] : 0;
        all = all && wave_max(left_over ? d[q] : 0) - wave_min(left_over ? d[q] : 0) <= 3;
        one = one && d[q] >= -1 && d[q] <= 1;
      }
      mine = all ? left_over : one;
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        lo[q] = wave_min(mine ? d[q] : 0);
        hi[q] = wave_max(mine ? d[q] : 0);
        r0[q] = h0[q] + lo[q] - 2;
        rs[q] = min(hi[q] - lo[q] + 5, A.nc[q]);
        const double u = frac_of(pi, q, A.flen) * A.nc[q] - cq[q] + d[q];
        bl[q] = wave_minf(mine ? u : (double)hi[q] + 1);
        bh[q] = wave_maxf(mine ? u : (double)lo[q]);
      }
    }
    todo &= ~__ballot(mine);
    const bool on = active && mine;
    WaveBox<real> wb, wv;
    wb.set(pi, A.box, lead, mine);
    if (has_v) wv.set(vi, A.box, lead, mine);
    // This wavefront's part of the cells, 64 at a time (lane t: the atom count
    // and start of cell q0 + t), or one range of the atoms as a single cell.
    // Their atoms are taken 64 at a time whatever the cells hold.
    const int ncells = A.brute ? P : rs[0] * rs[1] * rs[2];
    const int qb = (part + 1) * ncells / P;
    int q0 = part * ncells / P, at0 = 0, total = -1, incl = 0, first = 0;  // total < 0: not opened yet
    bool done = false, again = true;
    while (again) {
      // ---- gather candidates into this wavefront's segment
      int m[2] = {0, 0};
      while (!done) {
        if (total < 0) {
          if (q0 >= qb) {
            done = true;
            break;
          }
          int count = 0, start = 0;
          if (A.brute) {
            start = (int)((long long)part * A.n / P);
            count = lane == 0 ? (int)((long long)(part + 1) * A.n / P) - start : 0;
          } else if (q0 + lane < qb) {
            const int qq = q0 + lane;
            const int x[3] = {r0[0] + qq % rs[0], r0[1] + (qq / rs[0]) % rs[1], r0[2] + qq / (rs[0] * rs[1])};
            double g2 = 0;
#pragma unroll
            for (int e = 0; e < 3; ++e) {
              const double a = x[e] - h0[e], w = A.nc[e];
              double g = fmax(a - bh[e], bl[e] - a - 1);
              g = fmin(g, fmin(fmax(a - w - bh[e], bl[e] - a + w - 1), fmax(a + w - bh[e], bl[e] - a - w - 1)));
              g = fmax(0.0, g) * A.csize[e];
              g2 += g * g;
            }
            if (g2 <= reach2) {
              const int k = morton3(wrapc(x[0], A.nc[0]), wrapc(x[1], A.nc[1]), wrapc(x[2], A.nc[2]));
              count = A.cell_count[k];
              start = A.cell_start[k];
            }
          }
          incl = count;
#pragma unroll
          for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(incl, o, 64);
            if (lane >= o) incl += y;
          }
          first = start - (incl - count);  // sorted index of the cell's atoms = first + number in the part
          total = __builtin_amdgcn_readlane(incl, 63);
          at0 = 0;
        }
        if (at0 >= total) {
          total = -1;
          q0 += 64;
          continue;
        }
        if (m[0] + m[1] + 64 > kSeg) break;  // the segment is full: test first
        const int at = at0 + lane;
        int t = 0;  // the cell that holds number `at`: how many end at or before it
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) t += __shfl(incl, t + o - 1, 64) <= at ? o : 0;
        const int j = __shfl(first, t, 64) + at;
        bool km = false, kv = false;
        if (at < total) {
          km = wb.dist2(A.pos[j], A.box, A.periodic) <= A.rm2;
          if (has_v) kv = wv.dist2(A.vpos[j], A.box, A.periodic) <= A.rv2;
        }
        // tested for both lists, or only for the longer one
        const bool k0 = v_longer ? km : (has_v ? kv : km), k1 = !k0 && (km || kv);
        const unsigned long long b0 = __ballot(k0), b1 = __ballot(k1), below = (1ull << lane) - 1;
        if (k0) seg[part][m[0] + __popcll(b0 & below)] = j;
        if (k1) seg[part][kSeg - 1 - m[1] - __popcll(b1 & below)] = j;
        m[0] += __popcll(b0);
        m[1] += __popcll(b1);
        at0 += 64;
      }
      if (lane < 2) segn[lane][part] = lane ? m[1] : m[0];
      if (threadIdx.x == 0) more = 0;
      __syncthreads();
      if (lane == 0 && !done) more = 1;
      // ---- the segments in part order, in groups of 64
      int tot[2] = {0, 0};
      for (int u = 0; u < P; ++u) {
        tot[0] += segn[0][u];
        tot[1] += segn[1][u];
      }
      const int ng0 = (tot[0] + 63) / 64, ng = ng0 + (tot[1] + 63) / 64;
      for (int g = part; g < ng; g += P) {
        const int end = g < ng0 ? 0 : 1;
        int at = (g - (end ? ng0 : 0)) * 64 + lane, w = 0, j = -1;
        if (at < (end ? tot[1] : tot[0])) {
          while (at >= segn[end][w]) at -= segn[end][w++];
          j = seg[w][end ? kSeg - 1 - at : at];
        }
        const bool test_m = end == 0 || !v_longer, test_v = has_v && (end == 0 || v_longer);
        if (j >= 0) {  // places past the last candidate keep an older record: masked below
          if (test_m) grp[part][lane] = A.pos[j];
          if (test_v) vgrp[part][lane] = A.vpos[j];
        }
        __builtin_amdgcn_wave_barrier();
        unsigned long long mk = 0, vk = 0;
        if (test_m) mk = near_bits<real>(pi, grp[part], A, A.rs2[0]);
        if (test_v) vk = near_bits<real>(vi, vgrp[part], A, A.rs2[1]);
        __builtin_amdgcn_wave_barrier();
        const unsigned long long valid = __ballot(j >= 0);
        mk = on ? mk & valid : 0ull;
        vk = on ? vk & valid : 0ull;
        // an atom is not its own neighbor: clear the bits of the group's
        // candidates that are among these 64 atoms
        for (unsigned long long own = __ballot(j >= 0 && (j >> 6) == blk); own; own &= own - 1) {
          const int t = __builtin_ctzll(own);
          if ((__builtin_amdgcn_readlane(j, t) & 63) == lane) {
            mk &= ~(1ull << t);
            vk &= ~(1ull << t);
          }
        }
        cm += __popcll(mk);
        cv += __popcll(vk);
        if (gbase + g < A.ngmax) {
          const size_t o = ((size_t)lb * A.ngmax + gbase + g) * 64 + lane;
          A.cand[o] = j;
          A.mask[o] = ulonglong2{mk, vk};
        }
      }
      gbase += ng;
      __syncthreads();
      again = more != 0;
      __syncthreads();  // `more` and the segments are free again
    }
  }
  // ---- counts of the 64 atoms, their largest, and the slab sizes
  csum[0][part][lane] = cm;
  csum[1][part][lane] = cv;
  __syncthreads();
  if (part < 2) {
    int a = 0;
    for (int u = 0; u < P; ++u) a += csum[part][u][lane];
    const int mx = wave_max(a);
    int* nl = part == 0 ? A.nm : A.nv;
    if (nl) {
      if (active) nl[s0] = a;
      if (lane == 0) {
        (part == 0 ? A.mm : A.mv)[blk] = mx;
        (part == 0 ? A.sm : A.sv)[blk] = 64LL * mx;
      }
    }
    if (part == 0 && lane == 0) A.ngroup[blk] = gbase;
  }
}

// Entries of the lists from the masks (even workgroups the multipole list, bit
// set x, odd ones the vdW list, bit set y): the lane's bits in candidate
// order, each with the scale class of the pair, at the lane's rows of the
// slab.  Groups go in batches of kFillGroups; their per-lane counts give each
// group's first row.  The wavefronts drop the bits' candidate numbers (16
// bits) into rows in LDS; the rows are then written whole, lane by lane the
// candidate's index and its class looked up on the way (an entry written by
// itself touches a row of its own in every lane, and a bit loop that also
// looked up classes was bound by its instructions: both lists of 96,000 atoms
// 674 -> 241 us).
struct FillArgs {
  const int* eoff;
  const int* ej;
  const int* ec;
  const long long* off;
  uint32_t* out;
};
constexpr int kFillGroups = 64, kFillRows = 440;
__global__ __launch_bounds__(64 * kParts) void k_nb_fill(int n, int wave0, int ngmax, int nlists,
                                                         const int* __restrict__ ngroup,
                                                         const int* __restrict__ cand,
                                                         const ulonglong2* __restrict__ mask,
                                                         const int* __restrict__ perm, const int* __restrict__ iperm,
                                                         FillArgs fm, FillArgs fv) {
  __shared__ unsigned short rows[kFillRows][64];
  __shared__ unsigned short first[kFillGroups][64];  // first row of each group, from the batch's
  __shared__ int cj[kFillGroups * 64];
  __shared__ int count_l[64];
  const int lane = threadIdx.x & 63, part = threadIdx.x >> 6;
  const int lb = xcd_block();
  const int wave = lb / nlists, which = lb - wave * nlists, blk = wave0 + wave;
  const FillArgs F = which ? fv : fm;
  const int s = blk * 64 + lane;
  const int ng = ngroup[blk];
  const size_t gb = (size_t)wave * ngmax * 64;
  auto bits = [&](int g) {
    const ulonglong2 m = mask[gb + (size_t)g * 64 + lane];
    return which ? m.y : m.x;
  };
  Partners px;
  {
    const int oi = s < n ? perm[s] : 0;
    px.load(s < n ? F.eoff[oi] : 0, s < n ? F.eoff[oi + 1] : 0, F.ej, F.ec, iperm);
  }
  const long long wb = F.off[blk];
  int base = 0;  // rows filled before this batch
  for (int g0 = 0; g0 < ng; g0 += kFillGroups) {
    const int nb = min(kFillGroups, ng - g0);
    for (int g = part; g < nb; g += kParts) {
      first[g][lane] = (unsigned short)__popcll(bits(g0 + g));
      cj[g * 64 + lane] = cand[gb + (size_t)(g0 + g) * 64 + lane];
    }
    __syncthreads();
    if (part == 0) {
      int run = 0;
      for (int g = 0; g < nb; g += 4) {
        int v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = g + u < nb ? first[g + u][lane] : 0;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if (g + u < nb) first[g + u][lane] = (unsigned short)run;
          run += v[u];
        }
      }
      count_l[lane] = run;
    }
    __syncthreads();
    const int tot = count_l[lane];
    const int lo = wave_min(base), hi = wave_max(base + tot);
    for (int r0 = lo; r0 < hi; r0 += kFillRows) {
      const int r1 = min(r0 + kFillRows, hi);
      for (int g = part; g < nb; g += kParts) {
        const unsigned long long m = bits(g0 + g);
        int k = base + first[g][lane];
        if (k >= r1 || k + __popcll(m) <= r0) continue;
        k -= r0;
#pragma unroll
        for (int h = 0; h < 2; ++h)
          for (unsigned w = (unsigned)(m >> (32 * h)); w; w &= w - 1) {
            if ((unsigned)k < (unsigned)(r1 - r0)) rows[k][lane] = (unsigned short)(g * 64 + 32 * h + __builtin_ctz(w));
            ++k;
          }
      }
      __syncthreads();
      if (s < n) {
        const int k1 = min(r1, base + tot);
        for (int r = max(r0, base), q = r + ((part - (r - r0)) & (kParts - 1)); q < k1; q += kParts) {
          const int j = cj[rows[q - r0][lane]];
          F.out[wb + (long long)q * 64 + lane] = ((uint32_t)j << kCodeBits) | (uint32_t)px.find(j);
        }
      }
      __syncthreads();
    }
    base += tot;
  }
}

// Displacement check: any atom that moved more than half the list buffer
// since the last build writes `stamp` (a new value per check) to the flag, so
// the flag needs no clearing between checks.
template <class real>
__global__ void k_max_disp(int n, const double* __restrict__ xyz, const double* __restrict__ last, double lx,
                           double ly, double lz, int periodic, double lim2, int stamp, int* __restrict__ flag) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double dx = xyz[3 * i] - last[3 * i], dy = xyz[3 * i + 1] - last[3 * i + 1], dz = xyz[3 * i + 2] - last[3 * i + 2];
  if (periodic) {
    dx -= lx * rint(dx / lx);
    dy -= ly * rint(dy / ly);
    dz -= lz * rint(dz / lz);
  }
  if (dx * dx + dy * dy + dz * dz > lim2) *flag = stamp;
}


void list_capacity(NbList& L, long long total) {
  if ((size_t)total > L.capacity || !L.entries.p) {
    size_t cap = (size_t)(total * 1.2) + 64 * 64;
    L.entries.alloc(sizeof(uint32_t) * cap);
    L.capacity = cap;
  }
  L.total = total;
}

// Both lists from the candidate cells: masks and counts, offsets, entries.
// The masks have room for list_groups groups per wave (from the previous
// build; 64, 4,096 candidates, for a context's first); a wave that found more
// has the scan repeated with room for them, for as many waves at a time as
// kMaskBytes hold (T9HIP_LISTS=tiny starts with 1 and repeats for 3 waves at a
// time).  Without cells every wave may find all n atoms, masks of 0.3 n^2 bytes
// in all (78 GB for 500,000 atoms in no spatial order).
constexpr size_t kMaskBytes = 4ull << 30, kGroupBytes = 64 * (sizeof(int) + sizeof(ulonglong2));
template <class real>
void build_lists(Ctx& c) {
  const int n = c.n, nw = c.nwave;
  const bool has_v = c.vlist.cutoff > 0;
  ListArgs<real> A;
  A.n = n;
  A.brute = c.brute ? 1 : 0;
  A.periodic = c.periodic ? 1 : 0;
  A.pos = c.pos.as<PosRec<real>>();
  A.vpos = has_v ? c.vpos.as<PosRec<real>>() : nullptr;
  A.cellc = c.cellc.as<int>();
  for (int d = 0; d < 3; ++d) {
    A.nc[d] = c.ncell[d];
    A.csize[d] = c.periodic ? c.box[d] / c.ncell[d] : 1.0;
    A.flen[d] = c.periodic ? c.box[d] : 1.0;
  }
  A.cell_start = c.cell_start.as<int>();
  A.cell_count = c.cell_count.as<int>();
  A.box = make_boxT<real>(c);
  A.rm2 = (real)(c.mlist.cutoff * c.mlist.cutoff);
  A.rv2 = has_v ? (real)(c.vlist.cutoff * c.vlist.cutoff) : (real)0;
  A.reach = c.cell_reach;
  A.rs2[0] = A.rm2;
  A.rs2[1] = A.rv2;
  if (sizeof(real) == 4) {
    const double q = A.box.q[0];
    A.sy = (real)(A.box.q[1] / q * (A.box.q[1] / q));
    A.sz = (real)(A.box.q[2] / q * (A.box.q[2] / q));
    for (real& r : A.rs2) r = (real)(r * (1.0 + 1e-6) / (q * q));
  }
  NbList* lists[2] = {&c.mlist, &c.vlist};
  for (NbList* L : lists)
    if (L->cutoff > 0) {
      L->nlist.alloc(sizeof(int) * n);
      L->maxlen.alloc(sizeof(int) * nw);
      L->off.alloc(sizeof(long long) * (nw + 1));
      L->slots.alloc(sizeof(long long) * nw);
    }
  A.nm = c.mlist.nlist.as<int>();
  A.mm = c.mlist.maxlen.as<int>();
  A.sm = c.mlist.slots.as<long long>();
  A.nv = has_v ? c.vlist.nlist.as<int>() : nullptr;
  A.mv = has_v ? c.vlist.maxlen.as<int>() : nullptr;
  A.sv = has_v ? c.vlist.slots.as<long long>() : nullptr;
  c.list_ngroup.alloc(sizeof(int) * nw);
  A.ngroup = c.list_ngroup.as<int>();
  c.list_tot.alloc(3 * sizeof(long long));
  long long* d_tot = c.list_tot.as<long long>();
  // the largest group count and the totals come back in one readback (pinned
  // slots 45 to 47)
  long long* h_tot = reinterpret_cast<long long*>(c.h_scalars + 45);
  const char* mode = std::getenv("T9HIP_LISTS");
  const bool tiny = mode && !std::strcmp(mode, "tiny");
  auto masks = [&](int wave0, int waves, int room) {
    const size_t slots = (size_t)waves * room * 64;
    if (sizeof(int) * slots > c.list_cand.bytes) c.list_cand.alloc(sizeof(int) * slots);
    if (sizeof(ulonglong2) * slots > c.list_mask.bytes) c.list_mask.alloc(sizeof(ulonglong2) * slots);
    A.wave0 = wave0;
    A.ngmax = room;
    A.cand = c.list_cand.as<int>();
    A.mask = c.list_mask.as<ulonglong2>();
    // two workgroups of 8 wavefronts share a CU, so that one tests while the
    // other gathers (96,000 atoms: 359 us, against 414 with one of 16); a
    // system with less than one workgroup per CU takes 16 (3,000 atoms: 70 us
    // against 85).  Whole builds with 16 and 8: 254 waves 200 and 252 us;
    // above the line it depends on how full the last round of workgroups is:
    // 258 waves 210 and 264, 375 211 and 191, 516 319 and 330, 750 386 and 396,
    // 1,022 512 and 493, 4,500 1,895 and 1,666
    if (nw > 256) hipLaunchKernelGGL((k_nb_masks<real, 8>), dim3(waves), dim3(64 * 8), 0, c.stream, A);
    else hipLaunchKernelGGL((k_nb_masks<real, 16>), dim3(waves), dim3(64 * 16), 0, c.stream, A);
    T9_LAUNCH_CHECK();
  };
  int room = tiny ? 1 : c.list_groups;
  masks(0, nw, room);
  hipLaunchKernelGGL(k_list_totals, dim3(has_v ? 3 : 2), dim3(kScanBlock), 0, c.stream, nw, A.ngroup, A.sm,
                     c.mlist.off.as<long long>(), A.sv, has_v ? c.vlist.off.as<long long>() : nullptr, d_tot);
  T9_LAUNCH_CHECK();
  T9_HIP(hipMemcpyAsync(h_tot, d_tot, 3 * sizeof(long long), hipMemcpyDeviceToHost, c.stream));
  mark_readback(c);
  wait_marked(c);
  // the counts are whole whatever the masks had room for
  for (int q = 0; q < 2; ++q)
    if (lists[q]->cutoff > 0 && (h_tot[1 + q] < 0 || h_tot[1 + q] > (1LL << 31)))
      throw ListOverflow("neighbor list exceeds 2^31 slots");
  for (int q = 0; q < 2; ++q)
    if (lists[q]->cutoff > 0) list_capacity(*lists[q], h_tot[1 + q]);
  const bool repeat = h_tot[0] > room;
  int step = nw;  // waves at a time
  if (repeat) {
    room = (int)h_tot[0];
    step = tiny ? 3 : (int)std::min<size_t>(nw, std::max<size_t>(1, kMaskBytes / (room * kGroupBytes)));
  }
  c.list_groups = (int)std::max<size_t>(64, std::min<size_t>(h_tot[0] + h_tot[0] / 8, kMaskBytes / (nw * kGroupBytes)));
  const FillArgs fm{c.excl_off.as<int>(), c.excl_j.as<int>(), c.excl_code.as<int>(), c.mlist.off.as<long long>(),
                    c.mlist.entries.as<uint32_t>()};
  FillArgs fv = fm;
  if (has_v)
    fv = FillArgs{c.vexcl_off.as<int>(), c.vexcl_j.as<int>(), c.vexcl_code.as<int>(), c.vlist.off.as<long long>(),
                  c.vlist.entries.as<uint32_t>()};
  const int nlists = has_v ? 2 : 1;
  for (int w0 = 0; w0 < nw; w0 += step) {
    const int waves = std::min(step, nw - w0);
    if (repeat) masks(w0, waves, room);
    hipLaunchKernelGGL(k_nb_fill, dim3(waves * nlists), dim3(64 * kParts), 0, c.stream, n, w0, room, nlists, A.ngroup,
                       A.cand, A.mask, c.perm.as<int>(), c.iperm.as<int>(), fm, fv);
    T9_LAUNCH_CHECK();
  }
}

template <class real>
void nblist_build_t(Ctx& c) {
  const int n = c.n;
  const int nb = ceil_div(n, 256);
  if (c.brute) {  // no cells: caller order
    hipLaunchKernelGGL(k_identity, dim3(nb), dim3(256), 0, c.stream, n, c.perm.as<int>());
    T9_LAUNCH_CHECK();
  } else {
    const int nkeys = 1 << (3 * c.morton_bits);
    const int nchunk = ceil_div(nkeys, kScanBlock);
    c.cell_key.alloc(sizeof(int) * n);
    c.cell_rank.alloc(sizeof(int) * n);
    c.cell_count.alloc(sizeof(int) * nkeys);
    c.cell_start.alloc(sizeof(int) * nkeys);
    c.cell_csum.alloc(sizeof(int) * nchunk);
    c.unsorted.alloc(sizeof(int) * n);
    c.cellc_orig.alloc(sizeof(int) * n);
    T9_HIP(hipMemsetAsync(c.cell_count.p, 0, sizeof(int) * nkeys, c.stream));
    hipLaunchKernelGGL(k_cell_assign, dim3(nb), dim3(256), 0, c.stream, n, c.xyz.as<double>(), c.box[0], c.box[1],
                       c.box[2], c.ncell[0], c.ncell[1], c.ncell[2], c.cell_key.as<int>(), c.cell_rank.as<int>(),
                       c.cell_count.as<int>(), c.cellc_orig.as<int>());
    T9_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_count_sums, dim3(nchunk), dim3(kScanBlock), 0, c.stream, c.cell_count.as<int>(),
                       c.cell_csum.as<int>(), nkeys);
    hipLaunchKernelGGL(k_count_scan, dim3(nchunk), dim3(kScanBlock), 0, c.stream, c.cell_count.as<int>(),
                       c.cell_csum.as<int>(), c.cell_start.as<int>(), nkeys);
    T9_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_cell_scatter, dim3(nb), dim3(256), 0, c.stream, n, c.cell_key.as<int>(),
                       c.cell_rank.as<int>(), c.cell_start.as<int>(), c.unsorted.as<int>());
    T9_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_cell_sort, dim3(ceil_div(nkeys, 4)), dim3(256), 0, c.stream, nkeys,
                       c.cell_start.as<int>(), c.cell_count.as<int>(), c.unsorted.as<int>(), c.perm.as<int>());
    T9_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_build_sorted<real>, dim3(nb), dim3(256), 0, c.stream, n, c.perm.as<int>(), c.iperm.as<int>(),
                     c.xyz.as<double>(), c.xyz_last.as<double>(), make_double3(c.vorg[0], c.vorg[1], c.vorg[2]),
                     make_double3(c.vlen[0], c.vlen[1], c.vlen[2]), c.periodic ? 1 : 0,
                     c.pos.as<PosRec<real>>(), c.brute ? nullptr : c.cellc_orig.as<int>(), c.cellc.as<int>(),
                     c.polarity_o.as<double>(), c.pdamp_o.as<double>(), c.jpolar_o.as<int>(), c.polarity.as<real>(),
                     c.polinv.as<real>(), c.pdamp.as<real>(), c.jpolar.as<int>());
  T9_LAUNCH_CHECK();
  if (c.vlist.cutoff > 0) vdw_sites(c);
  build_lists<real>(c);
  c.builds++;
  c.list_valid = true;
  c.coords_dirty = false;
  c.rpole_valid = false;
  c.bins_valid = false;
  c.mlist.cut_valid = false;
}

// Keep the entries within the interaction cutoff (same FP arithmetic as the
// pair kernels, so those kernels need no distance test of their own), in
// list order (which keeps the pair kernels' gathers spatially local); with
// cut2b > 0 also the entries within the shorter second radius into
// ecut2 / ncut2, same layout.  kPairParts wavefronts per 64 atoms: in each
// round the wavefronts take consecutive, wave-uniform chunks of C <= 64 list
// positions (so a load instruction reads one contiguous 256-byte row) and
// record which entries fall inside each radius in 64-bit masks; the per-part
// counts are summed in part order through LDS, and each part then places its
// kept entries from its offset on.  The output slab of the 64 atoms is
// assembled in LDS (the first kCompactRowsA / kCompactRowsB rows; later rows,
// rare, go straight to memory) and written as whole 256-byte rows: written
// entry by entry, every store of a wavefront would touch 64 different rows.

template <class real>
__global__ __launch_bounds__(64 * kPairParts) void k_compact_parts(
    int n, const int* __restrict__ nlist, const long long* __restrict__ woff, const uint32_t* __restrict__ entries,
    const PosRec<real>* __restrict__ pos, BoxT<real> box, real cut2, real cut2b, int* __restrict__ ncut,
    uint32_t* __restrict__ ecut, int* __restrict__ ncut2, uint32_t* __restrict__ ecut2) {
  constexpr int P = kPairParts;
  __shared__ unsigned short cnt_a[P][64], cnt_b[P][64];
  __shared__ uint32_t rows_a[kCompactRowsA][64], rows_b[kCompactRowsB][64];
  const int part = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int blk = xcd_block();
  const int s = blk * 64 + lane;
  const bool two = ecut2 != nullptr;
  const bool valid = s < n;
  const int len = valid ? nlist[s] : 0;
  const int maxlen = wave_max(len);
  const long long base = woff[blk] + lane;
  const uint32_t* e = entries + base;
  PosRec<real> pi;
  if (valid) pi = pos[s];
  int tot_a = 0, tot_b = 0;  // kept entries of this atom in earlier rounds
  for (int k0 = 0; k0 < maxlen;) {
    const int C = min(64, (maxlen - k0 + P - 1) / P);
    const int kb = k0 + part * C;
    const int ke = min(kb + C, len);
    unsigned long long ma = 0, mb = 0;
    for (int k0 = kb; k0 < ke; k0 += 8) {  // 8 entries, then their 8 partners, in flight
      uint32_t ent[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) ent[u] = k0 + u < ke ? e[(long long)(k0 + u) * 64] : 0u;
      PosRec<real> pj[8];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (k0 + u < ke) pj[u] = pos[ent[u] >> kCodeBits];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (k0 + u < ke) {
          real xr, yr, zr;
          pair_disp(pi, pj[u], box, xr, yr, zr);
          const real r2 = xr * xr + yr * yr + zr * zr;
          if (r2 <= cut2) ma |= 1ull << (k0 + u - kb);
          if (two && r2 <= cut2b) mb |= 1ull << (k0 + u - kb);
        }
    }
    cnt_a[part][lane] = (unsigned short)__popcll(ma);
    cnt_b[part][lane] = (unsigned short)__popcll(mb);
    __syncthreads();
    int oa = tot_a, ob = tot_b;
    for (int q = 0; q < P; ++q) {
      if (q < part) {
        oa += cnt_a[q][lane];
        ob += cnt_b[q][lane];
      }
      tot_a += cnt_a[q][lane];
      tot_b += cnt_b[q][lane];
    }
    __syncthreads();
    while (ma | mb) {
      const int ja = ma ? __ffsll((long long)ma) - 1 : 64, jb = mb ? __ffsll((long long)mb) - 1 : 64;
      const int j = min(ja, jb);
      const uint32_t ent = e[(long long)(kb + j) * 64];
      if (j == ja) {
        if (oa < kCompactRowsA) rows_a[oa][lane] = ent;
        else ecut[base + (long long)oa * 64] = ent;
        ++oa;
        ma &= ma - 1;
      }
      if (j == jb) {
        if (ob < kCompactRowsB) rows_b[ob][lane] = ent;
        else ecut2[base + (long long)ob * 64] = ent;
        ++ob;
        mb &= mb - 1;
      }
    }
    k0 += P * C;
  }
  if (valid && part == 0) {
    ncut[s] = tot_a;
    if (two) ncut2[s] = tot_b;
  }
  // whole rows out; slots past an atom's count hold stale values that no
  // kernel reads (it reads positions below ncut)
  const int ra = min(wave_max(tot_a), kCompactRowsA), rb = two ? min(wave_max(tot_b), kCompactRowsB) : 0;
  __syncthreads();
  const long long wb = woff[blk];
  for (int q = threadIdx.x; q < ra * 64; q += 64 * P) ecut[wb + q] = rows_a[q >> 6][q & 63];
  for (int q = threadIdx.x; q < rb * 64; q += 64 * P) ecut2[wb + q] = rows_b[q >> 6][q & 63];
}

template <class real>
void compact_t(Ctx& c, hipStream_t st) {
  BoxT<real> box = make_boxT<real>(c);
  NbList* L = &c.mlist;
  if (!nblist_compact_buffers(c)) return;
  const bool two = L->cut2nd > 0;
  const double c2 = L->cut * L->cut, c2b = L->cut2nd * L->cut2nd;
  hipLaunchKernelGGL(k_compact_parts<real>, dim3(c.nwave), dim3(64 * kPairParts), 0, st, c.n,
                     L->nlist.as<int>(), L->off.as<long long>(), L->entries.as<uint32_t>(), c.pos.as<PosRec<real>>(),
                     box, (real)(c2 > 1e30 ? 1e30 : c2), (real)(two ? c2b : -1.0), L->ncut.as<int>(),
                     L->ecut.as<uint32_t>(), two ? L->ncut2.as<int>() : nullptr,
                     two ? L->ecut2.as<uint32_t>() : nullptr);
  T9_LAUNCH_CHECK();
  L->cut_valid = true;
}

template <class real>
void refresh_kernels_t(Ctx& c);

template <class real>
bool needs_rebuild_t(Ctx& c, bool refresh) {
  if (!c.list_valid) return true;
  if (!c.disp_flag.p) {  // allocated and cleared once; stamps start at 1
    c.disp_flag.alloc(sizeof(int));
    T9_HIP(hipMemsetAsync(c.disp_flag.p, 0, sizeof(int), c.stream));
  }
  const int stamp = c.disp_stamp = c.disp_stamp == INT_MAX ? 1 : c.disp_stamp + 1;
  double half = 0.5 * c.opt.list_buffer;
  hipLaunchKernelGGL(k_max_disp<real>, dim3(ceil_div(c.n, 256)), dim3(256), 0, c.stream, c.n, c.xyz.as<double>(),
                     c.xyz_last.as<double>(), c.box[0], c.box[1], c.box[2], c.periodic ? 1 : 0, half * half, stamp,
                     c.disp_flag.as<int>());
  T9_LAUNCH_CHECK();
  // read into pinned memory (a spare slot of the scalar readback buffer)
  int* h = reinterpret_cast<int*>(c.h_scalars + kDispSlot);
  T9_HIP(hipMemcpyAsync(h, c.disp_flag.p, sizeof(int), hipMemcpyDeviceToHost, c.stream));
  mark_readback(c);
  if (refresh) refresh_kernels_t<real>(c);  // runs while the host waits; a rebuild overwrites it
  wait_marked(c);
  return *h == stamp;
}

template <class real>
void refresh_kernels_t(Ctx& c) {
  hipLaunchKernelGGL(k_refresh_pos<real>, dim3(ceil_div(c.n, 256)), dim3(256), 0, c.stream, c.n, c.perm.as<int>(),
                     c.xyz.as<double>(), make_double3(c.vorg[0], c.vorg[1], c.vorg[2]),
                     make_double3(c.vlen[0], c.vlen[1], c.vlen[2]), c.periodic ? 1 : 0, c.pdamp_o.as<double>(),
                     c.pos.as<PosRec<real>>());
  T9_LAUNCH_CHECK();
  if (c.vlist.cutoff > 0) vdw_sites(c);
}

template <class real>
void refresh_t(Ctx& c) {
  refresh_kernels_t<real>(c);
  nblist_mark_refreshed(c);
}

}  // namespace

void nblist_mark_refreshed(Ctx& c) {
  c.coords_dirty = false;
  c.rpole_valid = false;
  c.bins_valid = false;
  c.mlist.cut_valid = false;
}

void nblist_build(Ctx& c) {
  if (c.prec == 32) nblist_build_t<float>(c);
  else nblist_build_t<double>(c);
}

bool nblist_needs_rebuild(Ctx& c, bool refresh) {
  return c.prec == 32 ? needs_rebuild_t<float>(c, refresh) : needs_rebuild_t<double>(c, refresh);
}

bool nblist_compact_buffers(Ctx& c) {
  NbList* L = &c.mlist;
  if (L->cutoff <= 0 || !L->entries.p) return false;
  L->ncut.alloc(sizeof(int) * c.n);
  L->ecut.alloc(sizeof(uint32_t) * L->capacity);
  if (L->cut2nd > 0) {
    L->ncut2.alloc(sizeof(int) * c.n);
    L->ecut2.alloc(sizeof(uint32_t) * L->capacity);
  }
  return true;
}

void nblist_compact(Ctx& c, hipStream_t st) {
  if (!st) st = c.stream;
  if (c.prec == 32) compact_t<float>(c, st);
  else compact_t<double>(c, st);
}

void refresh_sorted_coords(Ctx& c) {
  if (c.prec == 32) refresh_t<float>(c);
  else refresh_t<double>(c);
}

}  // namespace t9
