// Immersed-boundary multi-direct-forcing kernels for gfx950 (FP64).
//
// Data model.  Every marker m owns 64 stencil entries e = 64*m + s with
// s = 16*ix + 4*iy + iz in the reference's x-outer, y, z-inner loop order
// (Solidbody.f90:1009-1015).  The cells those entries touch form the "band".
// Each band cell keeps its entries in ascending e, which is the order in
// which the reference's serial loops over markers (Solidbody.f90:1034-1048,
// 968-977) update a cell; a per-cell sequential reduction over its entries
// therefore rounds exactly as the reference does, with no atomics on values.
//
// The whole structure is built on the device each coupling call, with no
// global sort: k_ibm_stencil (one wave per marker) forms the stencil and
// counts every entry into its cell in the cell map, which gives the entry a
// slot; k_ibm_claim gives each cell's first entry a band number and the cell
// its range of the entry list (both from one atomic counter, so the band's
// order varies from call to call while every per-cell result does not);
// k_ibm_fill gives every entry its band cell and places the entries in arrival
// order, and k_ibm_rank moves each to its rank by e among its cell's entries.
// Five launches (seven with bids for the cells, counts per band cell and a
// scan of them), since each costs its launch and a trip to memory: kernels of
// 144 markers 34 -> 26 us and two launch gaps, of 2304 markers beside a bulk
// collide 76 -> 66 us.
// Band arrays
// have a fixed stride `cap` = 64*M (an upper bound of the band size) and the
// band size itself lives in device memory (ctl[kNband]), so nothing is read
// back between the kernels.
#pragma once
#include "fsil_common.h"
#include "fsil_lbm_kernels.h"

namespace fsil {

// control words of the coupling kept in device memory
enum IbmCtl {
  kBoxLo = 0,      // [0..2] lowest band cell coordinate per axis (the fluid kernels look
  kBoxHi = 3,      // [3..5] highest       up the cell map only inside this box)
  kNband = 6,      // number of band cells
  kErr = 7,        // first failing marker (1-based) * 4 + reason, INT_MAX when none (2: a late
                   // workgroup of k_couple, 3: not a number, 4: inconsistent band build)
  kDone = 8,       // multi-direct-forcing loop finished
  kIters = 9,      // iterations run
  kWarm = 10,      // learned warm start in use for this call
  kFallback = 11,  // 1: the warm start did not lower the residual, restart from zero; 2: restarted
  kDone0 = 12,     // the done word at the start of a loop (no iteration at all)
  kArrived = 13,   // workgroups of k_couple that reached its barriers so far (0 between calls)
  kRan = 14,       // the last forcing round whose interpolation ran (-1: none)
  kGuess = 15,     // 1: the learned guess was applied in this call (kept on fallback)
  kSkip = 16,      // forcing rounds the applied guess stands for (0 without a guess)
  kListed = 17,    // workgroups of k_couple whose part of the entry lists is written (0 between calls)
  kNew = 18,       // band cells claimed so far in this call (becomes kNband)
  kNewEntries = 19,  // and their entries (one 64-bit counter with kNew)
  kCtlWords = 20
};

// whether an error word tells of a band build that did not complete (a late
// workgroup of k_couple, an inconsistent build): the cell map then holds more
// than the band's cells
__host__ __device__ constexpr bool band_build_failed(int err) { return err == 2 || err == 4; }

static_assert(kErr == kBandErrWord, "the fused kernels read the coupling error word at kBandErrWord");

// 4-point Peskin kernel (Solidbody.f90:822-833), FP64; sqrt is correctly rounded
__host__ __device__ inline double peskin4(double x) {
  const double r = fabs(x);
  if (r < 1.0) return (3.0 - 2.0 * r + sqrt(1.0 + 4.0 * r * (1.0 - r))) * 0.125;
  if (r < 2.0) return (5.0 - 2.0 * r - sqrt(-7.0 + 4.0 * r * (3.0 - r))) * 0.125;
  return 0.0;
}

// trimedindex (Solidbody.f90:834-866): 1-based indices i-1..i+2 wrapped or
// mirrored by the face codes; returns 0, or 1 (below the min face) / 2
// (beyond the max face) for an index the face code cannot place, in which
// case the index is clamped into the block so later kernels stay in bounds.
__host__ __device__ inline int trim4(int i, int nd, int *out, int bclo, int bchi) {
  int err = 0;
  for (int k = -1; k <= 2; ++k) {
    int v = i + k;
    if (v < 1) {
      if (bclo == BC_PERIODIC) v += nd;
      else if ((bclo == BC_SYMMETRIC || bclo == BC_WALL) && v == 0) v = 2;
      else if (bclo == BC_WALL_HALFWAY && v == 0) v = 1;
      else { err = err ? err : 1; v = 1; }
    } else if (v > nd) {
      if (bchi == BC_PERIODIC) v -= nd;
      else if ((bchi == BC_SYMMETRIC || bchi == BC_WALL) && v == nd + 1) v = nd - 1;
      else if (bchi == BC_WALL_HALFWAY && v == nd + 1) v = nd;
      else { err = err ? err : 2; v = nd; }
    }
    if (v < 1 || v > nd) { err = err ? err : (v < 1 ? 1 : 2); v = v < 1 ? 1 : nd; }
    out[k + 1] = v;
  }
  return err;
}

// reset of the control words; clears the previous band from the cell map and
// the marker forces
__global__ __launch_bounds__(256) void k_ibm_reset(int *__restrict__ ctl, const long long *__restrict__ prev_cell,
                                                   int *__restrict__ cellmap, double *__restrict__ dstate,
                                                   int done0, int warm, int skip,
                                                   double *__restrict__ Eforce, int n3M) {
  const int nprev = ctl[kNband];
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nprev; i += gridDim.x * blockDim.x)
    cellmap[prev_cell[i]] = -1;
  // v_Eforce = 0 (Solidbody.f90:889)
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n3M; i += gridDim.x * blockDim.x) Eforce[i] = 0.0;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    ctl[kNew] = 0;
    ctl[kNewEntries] = 0;
    ctl[kRan] = -1;
    ctl[kErr] = 0x7fffffff;
    ctl[kDone] = done0;
    // a learned guess stands for the first `skip` forcing rounds: the loop
    // count continues from there
    ctl[kIters] = warm ? skip : 0;
    ctl[kWarm] = warm;
    ctl[kGuess] = warm;
    ctl[kSkip] = warm ? skip : 0;
    ctl[kFallback] = 0;
    ctl[kDone0] = done0;
    dstate[0] = 1e10;  // dmax before the first iteration (Solidbody.f90:893)
  }
}

struct StencilArgs {
  int M;
  const double *__restrict__ Exyz;       // 3*M
  const int *__restrict__ first_marker;  // per marker: first marker of its body
  double org[3];
  double dh, invdh;
  int nd[3];
  int bc[6];
  float *__restrict__ Ew;                // 12*M
  unsigned *__restrict__ keys;           // 64*M: cell of entry e = 64*m + s
  int *__restrict__ ctl;
  int *__restrict__ cellmap;             // entries per cell so far: -1 - their number
  int *__restrict__ slot;                // 64*M: arrival number of the entry in its cell
};

// UpdateElmtInterp_ (Solidbody.f90:760-821), one wave per marker: every lane
// forms the marker's anchor (from its body's first marker) and trimmed 4x3
// indices, lanes 0..11 write the FP32 weights, lane s the cell of entry s, and
// counts the entry into the cell map, where a cell of n entries so far holds
// -1 - n (cells outside the band hold -1).
// Returns the error code of the indices; lanes 0..11 get weight s of the
// marker's 12 in wt.
__device__ __forceinline__ int stencil_entry(const StencilArgs &a, int m, int s, unsigned &key, float &wt) {
  const int m0 = a.first_marker[m];
  const int sel[3] = {s >> 4, (s >> 2) & 3, s & 3};
  int cidx[3];
  int err = 0;
  wt = 0.0f;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int ii = (int)floor((a.Exyz[3LL * m0 + k] - a.org[k]) * a.invdh);
    const double x0 = a.org[k] + (double)ii * a.dh;
    double off = (a.Exyz[3LL * m + k] - x0) * a.invdh;
    int idx = (int)floor(off);
    off = off - (double)idx;
    idx = idx + ii + 1;
    int ix[4];
    const int e = trim4(idx, a.nd[k], ix, a.bc[2 * k], a.bc[2 * k + 1]);
    if (e && !err) err = e;
    cidx[k] = ix[sel[k]];
    if ((s >> 2) == k) wt = (float)peskin4((double)((s & 3) - 1) - off);
  }
  key = ((unsigned)(cidx[0] - 1) * (unsigned)a.nd[1] + (unsigned)(cidx[1] - 1)) * (unsigned)a.nd[2] +
        (unsigned)(cidx[2] - 1);
  return err;
}

__global__ __launch_bounds__(256) void k_ibm_stencil(StencilArgs a) {
  const int s = threadIdx.x & 63;
  const int m = blockIdx.x * 4 + ((int)threadIdx.x >> 6);
  if (m >= a.M) return;
  unsigned key;
  float wt;
  const int err = stencil_entry(a, m, s, key, wt);
  if (s < 12) a.Ew[12LL * m + s] = wt;
  if (s == 0 && err) atomicMin(&a.ctl[kErr], (m + 1) * 4 + err);
  a.keys[64LL * m + s] = key;
  a.slot[64LL * m + s] = -1 - atomicSub(&a.cellmap[key], 1);
}

// Cell-map accesses of the band build go through device-scope atomics (the
// workgroups that count into, claim and look up one cell run on different XCDs).
__device__ __forceinline__ int cellmap_load(const int *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The first entry of each cell takes a band number and the cell's range of the
// entry list, whose start it leaves in ptr, and writes the number into the cell
// map.  One 1024-thread workgroup makes one atomic add on the counter of cells
// and entries (atomics on one line from many workgroups serialize): both are
// handed out together, so the ranges lie in band order.  The workgroup's part
// of the band's bounding box goes to blkbox[6 * workgroup ..] for k_ibm_fill.
constexpr int kClaimThreads = 1024;
__global__ __launch_bounds__(kClaimThreads) void k_ibm_claim(int E, const unsigned *__restrict__ keys,
                                                             const int *__restrict__ slot,
                                                             int *__restrict__ cellmap,
                                                             long long *__restrict__ band_cell,
                                                             int *__restrict__ ptr, int ny, int nz,
                                                             int *__restrict__ blkbox, int *__restrict__ ctl) {
  constexpr int NW = kClaimThreads / 64;
  __shared__ int wave_won[NW], wave_ent[NW], wave_off[NW], wave_eoff[NW], wbox[NW][6];
  __shared__ unsigned long long blk_base;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  const int s = threadIdx.x & 63, w = (int)threadIdx.x >> 6;
  const unsigned cell = e < E ? keys[e] : 0u;
  const bool won = e < E && slot[e] == 0;
  const int n = won ? -1 - cellmap_load(&cellmap[cell]) : 0;  // the cell's entries
  const unsigned long long mask = __ballot(won);
  int v[3];
  {
    const unsigned plane = (unsigned)ny * (unsigned)nz;
    const unsigned x = cell / plane, r = cell - x * plane, y = r / (unsigned)nz;
    v[0] = (int)x;
    v[1] = (int)y;
    v[2] = (int)(r - y * (unsigned)nz);
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    int lo = won ? v[k] : 0x7fffffff, hi = won ? v[k] : -1;
    for (int off = 32; off > 0; off >>= 1) {
      lo = min(lo, __shfl_xor(lo, off, 64));
      hi = max(hi, __shfl_xor(hi, off, 64));
    }
    if (s == 0) {
      wbox[w][k] = lo;
      wbox[w][3 + k] = hi;
    }
  }
  int upto = n;  // entries of the wave's cells up to this lane's
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(upto, off, 64);
    if (s >= off) upto += o;
  }
  if (s == 63) {
    wave_won[w] = __popcll(mask);
    wave_ent[w] = upto;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int t = 0, u = 0;
    for (int k = 0; k < NW; ++k) {
      wave_off[k] = t;
      wave_eoff[k] = u;
      t += wave_won[k];
      u += wave_ent[k];
    }
    blk_base = t ? atomicAdd(reinterpret_cast<unsigned long long *>(&ctl[kNew]),
                             ((unsigned long long)u << 32) | (unsigned long long)t)
                 : 0ULL;
  }
  if (threadIdx.x < 6) {
    const int k = threadIdx.x;
    int r = wbox[0][k];
    for (int q = 1; q < NW; ++q) r = k < 3 ? min(r, wbox[q][k]) : max(r, wbox[q][k]);
    blkbox[6 * blockIdx.x + k] = r;
  }
  __syncthreads();
  if (won) {
    const int b = (int)(blk_base & 0xffffffffULL) + wave_off[w] + __popcll(mask & ((1ULL << s) - 1ULL));
    band_cell[b] = (long long)cell;
    ptr[b] = (int)(blk_base >> 32) + wave_eoff[w] + upto - n;
    atomicExch(&cellmap[cell], b);
  }
}

__device__ __forceinline__ void band_macro_cell(const double *__restrict__ f, long long N, long long n, int b,
                                                int cap, double hv0, double hv1, double hv2,
                                                double *__restrict__ band_u);
__device__ __forceinline__ void band_macro32_cell(const float *__restrict__ g, long long N, long long n, int b,
                                                  int cap, double hv0, double hv1, double hv2,
                                                  double *__restrict__ band_u);

// the band velocity of the stored state (FP64 field f, or FP32 deviations g)
struct BandMacroArgs {
  const double *f;
  const float *g;
  long long N;
  const long long *cell;
  int cap;
  double hv0, hv1, hv2;
  double *band_u;
};

// every entry: its band cell, and its place in the cell's range in arrival
// order (k_ibm_rank restores entry order).  A cell without a band number or a
// place outside the list would be an inconsistent build: reported in ctl[kErr]
// (code 4), the entry skipped.
// Thread b < nband also forms band cell b's velocity from the stored state
// (k_band_macro's value).  The last workgroup reduces the claim workgroups'
// parts of the band's bounding box (nbox of them) into ctl[kBoxLo..kBoxHi+2]
// and closes the entry list.
__global__ __launch_bounds__(256) void k_ibm_fill(int E, const unsigned *__restrict__ keys,
                                                  const int *__restrict__ cellmap,
                                                  const int *__restrict__ slot, int *__restrict__ ptr,
                                                  int *__restrict__ bidx, int *__restrict__ tmp,
                                                  int *__restrict__ ctl, const int *__restrict__ blkbox, int nbox,
                                                  BandMacroArgs ma) {
  if (blockIdx.x == gridDim.x - 1) {
    __shared__ int wbox[4][6];
    const int lane = threadIdx.x & 63, w = (int)threadIdx.x >> 6;
    int r[6] = {0x7fffffff, 0x7fffffff, 0x7fffffff, -1, -1, -1};
    for (int q = threadIdx.x; q < nbox; q += blockDim.x)
#pragma unroll
      for (int k = 0; k < 6; ++k) r[k] = k < 3 ? min(r[k], blkbox[6 * q + k]) : max(r[k], blkbox[6 * q + k]);
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      int v = r[k];
      for (int off = 32; off > 0; off >>= 1) {
        const int o = __shfl_xor(v, off, 64);
        v = k < 3 ? min(v, o) : max(v, o);
      }
      if (lane == 0) wbox[w][k] = v;
    }
    __syncthreads();
    if (threadIdx.x < 6) {
      const int k = threadIdx.x;
      int v = wbox[0][k];
      for (int q = 1; q < 4; ++q) v = k < 3 ? min(v, wbox[q][k]) : max(v, wbox[q][k]);
      ctl[kBoxLo + k] = v;
    }
    if (threadIdx.x == 0) ptr[ctl[kNew]] = ctl[kNewEntries];
    return;
  }
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= E) return;
  const int b = cellmap_load(&cellmap[keys[e]]);
  const int sl = slot[e];
  if (e < ctl[kNew]) {
    if (ma.f) band_macro_cell(ma.f, ma.N, ma.cell[e], e, ma.cap, ma.hv0, ma.hv1, ma.hv2, ma.band_u);
    else band_macro32_cell(ma.g, ma.N, ma.cell[e], e, ma.cap, ma.hv0, ma.hv1, ma.hv2, ma.band_u);
  }
  const int at = b >= 0 && b < E && sl >= 0 ? ptr[b] + sl : -1;
  if (at < 0 || at >= E) {
    atomicMin(&ctl[kErr], 4);
    bidx[e] = 0;
    return;
  }
  bidx[e] = b;
  tmp[at] = e;
}

// every entry at its rank in its cell's range (the number of the cell's
// entries below it, its range read sixteen entries at a time), so each cell
// lists its entries in ascending e: went holds an entry's weights (rx, ry,
// rz) and its marker; the band size is published
__global__ __launch_bounds__(256) void k_ibm_rank(int E, int *__restrict__ ctl, const int *__restrict__ bidx,
                                                  const int *__restrict__ band_ptr, const int *__restrict__ tmp,
                                                  const float *__restrict__ Ew, float4 *__restrict__ went) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e == 0) ctl[kNband] = ctl[kNew];
  if (e >= E) return;
  // the entry's weights are read with its cell (they need nothing else)
  const int m = e >> 6, sidx = e & 63;
  const float *W = Ew + 12LL * m;
  const float wx = W[sidx >> 4], wy = W[4 + ((sidx >> 2) & 3)], wz = W[8 + (sidx & 3)];
  const int b = bidx[e];
  const int p0 = band_ptr[b], n = band_ptr[b + 1] - p0;
  int r = 0;
  for (int j0 = 0; j0 < n; j0 += 16) {
    int v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = j0 + j < n ? tmp[p0 + j0 + j] : 0x7fffffff;
#pragma unroll
    for (int j = 0; j < 16; ++j) r += v[j] < e ? 1 : 0;
  }
  // the entry's three stencil weights and its marker, in the cells' order
  // (an entry without a cell of its own, an error already reported, may not fit)
  if (r < n) went[p0 + r] = make_float4(wx, wy, wz, __int_as_float(m));
}

// band macros: den/u of every band cell from the stored state, same
// expressions as the collision kernel (FluidDomain.f90:1136-1139)
__device__ __forceinline__ void band_macro_cell(const double *__restrict__ f, long long N, long long n, int b,
                                                int cap, double hv0, double hv1, double hv2,
                                                double *__restrict__ band_u) {
  double g[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) g[q] = f[q * N + n];
  double s, m1, m2, m3;
  moments(g, s, m1, m2, m3);
  band_u[b] = (m1 + hv0) / s;
  band_u[cap + b] = (m2 + hv1) / s;
  band_u[2LL * cap + b] = (m3 + hv2) / s;
}

__global__ __launch_bounds__(256) void k_band_macro(const double *__restrict__ f, long long N,
                                                    const long long *__restrict__ cell,
                                                    const int *__restrict__ ctl, int cap,
                                                    double hv0, double hv1, double hv2,
                                                    double *__restrict__ band_u, int only_on_fallback = 0) {
  if (only_on_fallback && ctl[kFallback] != 1) return;
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= ctl[kNband]) return;
  band_macro_cell(f, N, cell[b], b, cap, hv0, hv1, hv2, band_u);
}

// band macros of the FP32-deviation state (the immersed-boundary coupling
// runs in FP64): rho = 1 + sum g, j = sum e g, summed in FP64 from the stored
// deviations
__global__ __launch_bounds__(256) void k_band_macro32(const float *__restrict__ g, long long N,
                                                      const long long *__restrict__ cell,
                                                      const int *__restrict__ ctl, int cap, double hv0,
                                                      double hv1, double hv2, double *__restrict__ band_u,
                                                      int only_on_fallback = 0) {
  if (only_on_fallback && ctl[kFallback] != 1) return;
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= ctl[kNband]) return;
  band_macro32_cell(g, N, cell[b], b, cap, hv0, hv1, hv2, band_u);
}

__device__ __forceinline__ void band_macro32_cell(const float *__restrict__ g, long long N, long long n, int b,
                                                  int cap, double hv0, double hv1, double hv2,
                                                  double *__restrict__ band_u) {
  double dr = 0.0, j1 = 0.0, j2 = 0.0, j3 = 0.0;
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const double v = (double)g[q * N + n];
    dr = dr + v;
    if (ex(q) != 0) j1 = ex(q) > 0 ? j1 + v : j1 - v;
    if (ey(q) != 0) j2 = ey(q) > 0 ? j2 + v : j2 - v;
    if (ez(q) != 0) j3 = ez(q) > 0 ? j3 + v : j3 - v;
  }
  const double rho = 1.0 + dr;
  band_u[b] = (j1 + hv0) / rho;
  band_u[cap + b] = (j2 + hv1) / rho;
  band_u[2LL * cap + b] = (j3 + hv2) / rho;
}

__global__ void k_zero(double *__restrict__ p, long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.0;
}

// every cell set to the same 19 populations (a uniform initial state)
struct Fill19 {
  double v[Q];
};
struct Fill19f {
  float v[Q];
};
__global__ __launch_bounds__(256) void k_fill19(double *__restrict__ f, long long N, Fill19 a) {
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
#pragma unroll
  for (int q = 0; q < Q; ++q) f[q * N + n] = a.v[q];
}
__global__ __launch_bounds__(256) void k_fill19f(float *__restrict__ g, long long N, Fill19f a) {
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
#pragma unroll
  for (int q = 0; q < Q; ++q) g[q * N + n] = a.v[q];
}

// plain copy (bandwidth calibration of the HBM counters and the roofline)
__global__ __launch_bounds__(256) void k_copy(const double *__restrict__ a, double *__restrict__ b,
                                              long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[i];
}

// wave64 sum through DPP/permute lanes (deterministic order)
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = v + __shfl_down(v, off, 64);
  return v;
}

// sum of tl[0..M) in a fixed order by one 256-thread workgroup: strided
// partial sums, a wave tree, then the four wave sums in order.  Each thread
// reads its terms sixteen at a time before adding them (in the same order),
// so the reads do not wait for one another; the first sixteen are read by
// the caller (mdf_tl_first), ahead of its other reads.
constexpr int kTlBatch = 16;
__device__ inline void mdf_tl_first(const double *tl, int M, double *v) {
  const int step = blockDim.x;
#pragma unroll
  for (int j = 0; j < kTlBatch; ++j) {
    const int m = (int)threadIdx.x + j * step;
    v[j] = m < M ? tl[m] : 0.0;
  }
}
__device__ inline double mdf_tl_sum(const double *tl, int M, const double *first) {
  constexpr int B = kTlBatch;
  double p = 0.0;
  const int step = blockDim.x;
  for (int base = threadIdx.x; base < M; base += B * step) {
    double v[B];
#pragma unroll
    for (int j = 0; j < B; ++j)
      v[j] = base == (int)threadIdx.x ? first[j] : (base + j * step < M ? tl[base + j * step] : 0.0);
#pragma unroll
    for (int j = 0; j < B; ++j)
      if (base + j * step < M) p = p + v[j];
  }
  __shared__ double part[4];
  p = wave_sum(p);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = p;
  __syncthreads();
  double tol = 0.0;
  for (int k = 0; k < (int)(blockDim.x + 63) / 64; ++k) tol = tol + part[k];
  return tol;
}

// stop test of the multi-direct-forcing loop (Solidbody.f90:895-906) from the
// summed |dV|_1 of the markers: dmax = tol / (sum M_b * Uref), one iteration
// counted; sets the done word when the loop condition fails.
// dstate[2] keeps the residual of loop iteration skip+1 (the first one after
// a learned guess standing for `skip` rounds) for the next call: a guessed
// call whose first residual exceeds twice that of the previous call restarts
// from the zero guess (k_ws_fallback, k_band_macro on fallback), which then
// runs the plain loop.  A negative dstate[2] (no previous call) always
// falls back.
// The words it reads, read up front (with the residual terms) so that the
// decision waits for no further reads.
struct MdfWords {
  int iters, warm, done0;
  double ref;
};
__device__ inline MdfWords mdf_words(const int *ctl, const double *dstate) {
  return MdfWords{ctl[kIters], ctl[kWarm], ctl[kDone0], dstate[2]};
}
__device__ inline void mdf_decide(int *ctl, double *dstate, double tol, double dsum, double Uref, int ntol,
                                  double dtol, int skip, const MdfWords &wd) {
  const int it = wd.iters + 1;
  ctl[kIters] = it;
  if (!isfinite(tol)) {
    atomicMin(&ctl[kErr], 3);  // "Nan found in PenaltyForce" (Solidbody.f90:1028-1031)
    ctl[kDone] = 1;
    return;
  }
  const double dm = tol / (dsum * Uref);
  dstate[0] = dm;
  if (it == skip + 1) {
    const double ref = wd.ref;
    dstate[2] = dm;
    if (wd.warm == 1 && !(ref >= 0.0 && dm <= 2.0 * ref)) {
      ctl[kWarm] = 0;
      ctl[kFallback] = 1;
      ctl[kIters] = 0;
      ctl[kDone] = wd.done0;
      dstate[0] = 1e10;
      return;
    }
  }
  if (!(it < ntol && dm > dtol)) ctl[kDone] = 1;
}

// One marker per wave: each lane forms one of the 64 interpolation terms
// ((u*rx)*ry)*rz of the marker's stencil (Solidbody.f90:1009-1015), lane 0
// adds them in the reference's x, y, z order, then the velocity defect,
// penalty force and force accumulation (PenaltyForce_, Solidbody.f90:1016-1026).
// The marker's |dV|_1 goes to tl[m] for the residual; ctl[kRan] = round
// records that this forcing round ran.
__global__ __launch_bounds__(256) void k_interp(int M, int round, const int *__restrict__ bidx,
                                                const float *__restrict__ Ew,
                                                const double *__restrict__ band_u, int cap,
                                                int *__restrict__ ctl,
                                                const double *__restrict__ Evel,
                                                const double *__restrict__ Ea, double invh3,
                                                double *__restrict__ Eforce,
                                                double *__restrict__ fT,
                                                double *__restrict__ tl, int snap = -1,
                                                double *__restrict__ Esnap = nullptr) {
  __shared__ double t[4][3][64];
  const int w = threadIdx.x >> 6, s = threadIdx.x & 63;
  const int m = blockIdx.x * 4 + w;
  // the stencil's band cells and weights and the marker's own values are read
  // with the control word (the reads are the kernel's latency)
  int b = 0;
  float wx = 0.0f, wy = 0.0f, wz = 0.0f;
  if (m < M) {
    b = bidx[64LL * m + s];
    const float *W = Ew + 12LL * m;
    wx = W[s >> 4];
    wy = W[4 + ((s >> 2) & 3)];
    wz = W[8 + (s & 3)];
  }
  double ev1 = 0.0, ev2 = 0.0, ev3 = 0.0, am = 0.0, ef1 = 0.0, ef2 = 0.0, ef3 = 0.0;
  if (m < M && s == 0) {
    ev1 = Evel[3LL * m]; ev2 = Evel[3LL * m + 1]; ev3 = Evel[3LL * m + 2];
    am = Ea[m];
    ef1 = Eforce[3LL * m]; ef2 = Eforce[3LL * m + 1]; ef3 = Eforce[3LL * m + 2];
  }
  if (ctl[kDone]) return;  // uniform over the grid
  if (blockIdx.x == 0 && threadIdx.x == 0) ctl[kRan] = round;
  if (m < M) {
    const double rx = (double)wx, ry = (double)wy, rz = (double)wz;
    t[w][0][s] = ((band_u[b] * rx) * ry) * rz;
    t[w][1][s] = ((band_u[cap + b] * rx) * ry) * rz;
    t[w][2][s] = ((band_u[2LL * cap + b] * rx) * ry) * rz;
  }
  __syncthreads();
  if (m < M && s == 0) {
    double v1 = 0.0, v2 = 0.0, v3 = 0.0;
#pragma unroll 16
    for (int k = 0; k < 64; ++k) {
      v1 = v1 + t[w][0][k];
      v2 = v2 + t[w][1][k];
      v3 = v3 + t[w][2][k];
    }
    const double d1 = ev1 - v1, d2 = ev2 - v2, d3 = ev3 - v3;
    const double F1 = d1 * am, F2 = d2 * am, F3 = d3 * am;
    tl[m] = (fabs(d1) + fabs(d2)) + fabs(d3);
    Eforce[3LL * m] = ef1 + F1;
    Eforce[3LL * m + 1] = ef2 + F2;
    Eforce[3LL * m + 2] = ef3 + F3;
    if (round == snap) {  // the force after round snap+1 (a training target of the warm start)
      Esnap[3LL * m] = ef1 + F1;
      Esnap[3LL * m + 1] = ef2 + F2;
      Esnap[3LL * m + 2] = ef3 + F3;
    }
    fT[3LL * m] = F1 * invh3;
    fT[3LL * m + 1] = F2 * invh3;
    fT[3LL * m + 2] = F3 * invh3;
  }
}

// The per-cell sums over a band cell's entries (the velocity correction and
// the spreading), by workgroups of 256 threads taking kCellsPerPass
// consecutive cells at a time: the cells' entries are one contiguous range of
// the CSR arrays, so each thread forms one entry's term from one coalesced
// read (weights and marker) and one gather (the marker's value) into LDS, and then one
// thread per cell adds its terms in entry order, as the sequential loop does.
// A pass whose range exceeds the LDS area (pass_cap <= kPassEntries entries)
// falls back to one thread per cell reading its entries itself.  SPREAD: term = -(((v h^-3 rx)
// ry) rz), g = sum + VF (out = band_F); else u -= ((v rx) ry) rz (out =
// band_u, read first).
constexpr int kCellsPerPass = 32;
constexpr int kPassEntries = 1024;  // 24 KiB of LDS: fits beside the bulk collide of a split step
template <bool SPREAD>
__device__ inline void band_cells_reduce(int blk, int nb, int nblk, int cap, const int *__restrict__ ptr,
                                         const float4 *__restrict__ went, const double *__restrict__ val,
                                         double invh3, double *__restrict__ out, double VF1, double VF2,
                                         double VF3, int pass_cap) {
  __shared__ int sptr[kCellsPerPass + 1];
  __shared__ double term[3][kPassEntries];
  const int t = threadIdx.x;
  for (int c0 = blk * kCellsPerPass; c0 < nb; c0 += nblk * kCellsPerPass) {
    const int nc = min(kCellsPerPass, nb - c0);
    double o1 = 0.0, o2 = 0.0, o3 = 0.0;
    if (t <= nc) sptr[t] = ptr[c0 + t];
    if (!SPREAD && t < nc) {
      o1 = out[c0 + t];
      o2 = out[cap + c0 + t];
      o3 = out[2LL * cap + c0 + t];
    }
    __syncthreads();
    const int e0 = sptr[0], ne = sptr[nc] - e0;
    const bool fits = ne <= pass_cap;
    if (fits) {
      for (int k = t; k < ne; k += blockDim.x) {
        const float4 w = went[e0 + k];
        const int m = __float_as_int(w.w);
        const double rx = (double)w.x, ry = (double)w.y, rz = (double)w.z;
        double v1 = val[3LL * m], v2 = val[3LL * m + 1], v3 = val[3LL * m + 2];
        if (SPREAD) {
          v1 = v1 * invh3; v2 = v2 * invh3; v3 = v3 * invh3;
          term[0][k] = -(((v1 * rx) * ry) * rz);
          term[1][k] = -(((v2 * rx) * ry) * rz);
          term[2][k] = -(((v3 * rx) * ry) * rz);
        } else {
          term[0][k] = ((v1 * rx) * ry) * rz;
          term[1][k] = ((v2 * rx) * ry) * rz;
          term[2][k] = ((v3 * rx) * ry) * rz;
        }
      }
    }
    __syncthreads();
    if (t < nc) {
      const int k0 = sptr[t] - e0, k1 = sptr[t + 1] - e0;
      for (int k = k0; k < k1; ++k) {
        double x1, x2, x3;
        if (fits) {
          x1 = term[0][k]; x2 = term[1][k]; x3 = term[2][k];
        } else {
          const float4 w = went[e0 + k];
          const int m = __float_as_int(w.w);
          const double rx = (double)w.x, ry = (double)w.y, rz = (double)w.z;
          double v1 = val[3LL * m], v2 = val[3LL * m + 1], v3 = val[3LL * m + 2];
          if (SPREAD) {
            v1 = v1 * invh3; v2 = v2 * invh3; v3 = v3 * invh3;
            x1 = -(((v1 * rx) * ry) * rz); x2 = -(((v2 * rx) * ry) * rz); x3 = -(((v3 * rx) * ry) * rz);
          } else {
            x1 = ((v1 * rx) * ry) * rz; x2 = ((v2 * rx) * ry) * rz; x3 = ((v3 * rx) * ry) * rz;
          }
        }
        if (SPREAD) {
          o1 = o1 + x1; o2 = o2 + x2; o3 = o3 + x3;
        } else {
          o1 = o1 - x1; o2 = o2 - x2; o3 = o3 - x3;
        }
      }
      if (SPREAD) {
        out[c0 + t] = o1 + VF1;
        out[cap + c0 + t] = o2 + VF2;
        out[2LL * cap + c0 + t] = o3 + VF3;
      } else {
        out[c0 + t] = o1;
        out[cap + c0 + t] = o2;
        out[2LL * cap + c0 + t] = o3;
      }
    }
    __syncthreads();  // (the next pass rewrites sptr and term)
  }
}

struct MdfTest {
  const double *tl;
  double *dstate;
  int M, ntol;
  double dsum, Uref, dtol;
  int skip;  // rounds a learned guess stands for (the fallback test is at iteration skip+1)
};

// velocity correction of every band cell: u -= fT*rx*ry*rz over its entries
// in (marker, stencil) order (Solidbody.f90:1034-1048), by the first
// cell_blocks workgroups (band_cells_reduce; the host sizes the grid to the
// last call's band).
// round >= 0: the correction of that forcing round (runs when its k_interp
// ran), and workgroup cell_blocks makes the round's stop test (the markers'
// |dV|_1 summed in a fixed order, then mdf_decide); round < 0 (the
// warm-start guess): runs unless the loop is done, no stop test.
__global__ __launch_bounds__(256) void k_correct(int *__restrict__ ctl, int round, MdfTest mt, int cap,
                                                 const int *__restrict__ ptr,
                                                 const float4 *__restrict__ went,
                                                 const double *__restrict__ fT,
                                                 double *__restrict__ band_u, int cell_blocks, int pass_cap) {
  if ((int)blockIdx.x >= cell_blocks) {
    // the stop test: its reads issued together, then the sums
    double first[kTlBatch];
    mdf_tl_first(mt.tl, mt.M, first);
    const MdfWords wd = mdf_words(ctl, mt.dstate);
    if (round >= 0 ? ctl[kRan] != round : ctl[kDone] != 0) return;  // uniform over the grid
    if (round >= 0) {
      const double tol = mdf_tl_sum(mt.tl, mt.M, first);
      if (threadIdx.x == 0) mdf_decide(ctl, mt.dstate, tol, mt.dsum, mt.Uref, mt.ntol, mt.dtol, mt.skip, wd);
    }
    return;
  }
  if (round >= 0 ? ctl[kRan] != round : ctl[kDone] != 0) return;  // uniform over the grid
  band_cells_reduce<false>(blockIdx.x, ctl[kNband], cell_blocks, cap, ptr, went, fT, 1.0, band_u, 0.0, 0.0, 0.0,
                           pass_cap);
}

// The band build and all forcing rounds of a call in one launch, one wave per
// marker, for marker counts whose workgroups are all resident at once
// (kCoupleShare); k_ibm_reset .. k_ibm_rank and the rounds' launches otherwise.
// Build: the launches' steps with a barrier between them, an entry's values
// staying in its lane's registers (marker m's wave, lane s: entry 64 m + s).
// Rounds: the lane holds the velocity of its entry's band cell and the cell's
// entries (weights and markers, the first kCoupleEntries of them in registers),
// so a cell's correction is formed by the wave of every marker whose stencil
// holds it and the only values that cross workgroups are the markers' forces and
// residual terms: a round is one exchange behind one barrier.  Every sum is
// formed in the order of k_interp, band_cells_reduce and mdf_tl_sum, and every
// workgroup makes the same stop test; workgroup 0 records it.
// What one workgroup writes and another reads in this launch goes through
// device-scope atomics (the workgroups run on several XCDs) and is complete
// before the writer is counted at the next barrier.  The barriers share one
// running count, so every workgroup waits at each of them: one that went on
// would be counted for the next barrier in place of a workgroup that has yet to
// reach this one.  The entry lists, for which only workgroups with a cell of
// more than kCoupleEntries entries wait, are counted in a word of their own.
// The rounds' exchange has two copies taken in turn: a workgroup writes round
// r+2's values only after all have passed barrier r+1, that is, have read round
// r's.
// A wait is bounded by kCoupleWait; the call then fails, k_ibm_finish leaves
// an empty band and the host clears the cell map, whose counts and numbers no
// longer match the band, and takes the launches from then on.
// Bound by the barriers and one wave's FP64 rate: 4.2 us per round (ordered sums
// 1.0, barrier 1.6, values into LDS and the residual 0.8, correction 0.8) where
// two launches took 9.7; the build 23 us (five barriers of 2, the stencil and
// stored state 4, claim 2.4, placing 3) where its launches took 26 and five gaps.
// Ten rounds of 144 markers with the build 68 us (launches: 123 and the gaps),
// three rounds of 256 42 us.  A whole coupling call of markers 0.9 x 0.7 cells
// apart, launches / one launch: 188 / 144 us (256 markers), 197 / 182 (512); with
// 512 markers in a few cells 1637 / 795.
struct CoupleArgs {
  StencilArgs st;  // (keys, slot and Ew are not used)
  BandMacroArgs ma;
  long long *cell;  // the band's cells, first the previous call's
  int *ptr, *tmp;
  float4 *went;
  const double *Evel, *Ea;
  double invh3;
  double *Eforce;
  double *xch;  // [2][4][M]: h^-3 F dt / (2 rho) per axis, |dV|_1
  MdfTest mt;
  int give_up;  // the barrier whose waits fail at once (0: none; for tests)
};

constexpr int kCoupleThreads = 256;   // four markers per workgroup
constexpr int kCoupleEntries = 16;    // entries of a cell held in registers (a plane of markers a cell apart: all)
// Every workgroup of the launch waits for every other, so all have to be
// resident together: at most half as many as the CUs, of which each holds two,
// so the launches of a process's four hardware queues fit at once, and other
// kernels beside them end by themselves.  The repeated corrections grow with
// the markers per workgroup's share of a CU; at the line (512 markers on 256
// CUs) the form is still the faster one.
constexpr int kCoupleShare = 2;
// On large blocks the collision beside the call is the longer chain, and this
// launch's workgroups keep CU slots from it.  us per step, launches / one
// launch, 225 markers, ten rounds and four beam sub-steps: 3.5M cells FP64 464 /
// 405, FP32 367 / 307; 5.9M 540 / 478 and 387 / 326; 9.7M 741 / 744 and 495 /
// 496.  Rigid, three rounds: 3.5M 265 / 249 and 172 / 157; 5.9M 376 / 383 and
// 245 / 244; 9.7M 641 / 639 and 383 / 384.  The line lies where a flexible body
// still gains 11-16%; a rigid one has lost its gain there.
constexpr long long kCoupleCells = 6LL << 20;
constexpr int kCoupleMarkers = 512;   // (the exchanged values are kept in LDS)
constexpr long long kCoupleWait = 1000000000LL;  // ticks of the 100 MHz clock: 10 s

template <class T>
__device__ __forceinline__ T xload(const T *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void xstore(T *p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Arrival: this workgroup's stores have reached memory, then it is counted.
// The wait ends when all workgroups are counted for the nth time (from 1: true),
// which holds only if none can be counted for nth + 1 before that, or late
// (false).
struct CoupleLate {  // (LDS)
  int give_up, late;
};
__device__ __forceinline__ void couple_arrive(int *arrived) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_fetch_add(arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool couple_wait(int *arrived, int nth, CoupleLate *c) {
  if (threadIdx.x == 0) {
    const int want = (int)gridDim.x * nth;
    const long long t0 = (long long)wall_clock64();
    const bool give_up = nth == c->give_up;
    while (give_up || xload(arrived) < want) {
      if (give_up || (long long)wall_clock64() - t0 > kCoupleWait) {
        c->late = 1;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
  }
  __syncthreads();
  return c->late == 0;
}
__device__ __forceinline__ bool couple_barrier(int *arrived, int nth, CoupleLate *c) {
  couple_arrive(arrived);
  return couple_wait(arrived, nth, c);
}

// ascending sort of sixteen values in registers (odd-even merges)
__device__ __forceinline__ void sort16(int *v) {
#pragma unroll
  for (int lp = 0; lp < 4; ++lp)
#pragma unroll
    for (int lk = lp; lk >= 0; --lk)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int p = 1 << lp, k = 1 << lk, lo = k % p;  // (compare i and i + k where both lie in one 2p block)
        if (i >= lo && (i - lo) % (2 * k) < k && i + k < 16 && i / (2 * p) == (i + k) / (2 * p)) {
          const int x = min(v[i], v[i + k]), y = max(v[i], v[i + k]);
          v[i] = x;
          v[i + k] = y;
        }
      }
}

// lane `l`'s value (l a constant)
__device__ __forceinline__ double lane_value(double v, int l) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), l), hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
  return __hiloint2double(hi, lo);
}

__global__ __launch_bounds__(kCoupleThreads, 2) void k_couple(CoupleArgs a) {
  constexpr int NW = kCoupleThreads / 64, B = kCoupleEntries;
  // the weights of all markers while the entry lists are made, then the
  // interpolation terms and the exchanged values
  __shared__ union {
    float W[kCoupleMarkers][12];
    struct {
      double t[NW][3][64], fx[4][kCoupleMarkers + 1];  // (value M: zero)
    } r;
  } lds;
  double(&t)[NW][3][64] = lds.r.t;
  double(&fx)[4][kCoupleMarkers + 1] = lds.r.fx;
  __shared__ double part[4];
  __shared__ int wave_won[NW], wave_ent[NW], wbox[NW][6];
  __shared__ CoupleLate late;
  __shared__ unsigned long long blk_base;
  const int w = threadIdx.x >> 6, s = threadIdx.x & 63;
  const int m = blockIdx.x * NW + w;
  const int M = a.st.M, E = 64 * M;
  const bool on = m < M;
  const int me = on ? m : M - 1;  // (a spare wave follows the last marker and stores nothing)
  const int e = 64 * me + s;
  int *const ctl = a.st.ctl, *const cellmap = a.st.cellmap, *const arrived = &ctl[kArrived];
  const bool first = blockIdx.x == 0 && threadIdx.x == 0;
  if (threadIdx.x == 0) late = CoupleLate{a.give_up, 0};
  // k_ibm_reset's work
  {
    const int nprev = ctl[kNband];
    for (int i = blockIdx.x * kCoupleThreads + threadIdx.x; i < nprev; i += gridDim.x * kCoupleThreads)
      xstore(&cellmap[a.cell[i]], -1);
    const int k = threadIdx.x;
    if (blockIdx.x == 0 && k < kCtlWords && k != kNband && k != kArrived && k != kListed)
      xstore(&ctl[k], k < 3 || k == kErr ? 0x7fffffff : k < 6 || k == kRan ? -1 : 0);
    if (first) a.mt.dstate[0] = 1e10;
  }
  unsigned key;
  float wt;
  const int err = stencil_entry(a.st, me, s, key, wt);
  if (on && s < 12) xstore(&a.st.Ew[12LL * m + s], wt);
  const float fwx = __shfl(wt, s >> 4, 64), fwy = __shfl(wt, 4 + ((s >> 2) & 3), 64),
              fwz = __shfl(wt, 8 + (s & 3), 64);
  double u[3];
  if (a.ma.f) band_macro_cell(a.ma.f, a.ma.N, key, 0, 1, a.ma.hv0, a.ma.hv1, a.ma.hv2, u);
  else band_macro32_cell(a.ma.g, a.ma.N, key, 0, 1, a.ma.hv0, a.ma.hv1, a.ma.hv2, u);
  const int c = min(s, 2);  // lane c < 3: component c of the marker
  const double ev = a.Evel[3LL * me + c], am = a.Ea[me];
  const double ref = a.mt.dstate[2];
  if (!couple_barrier(arrived, 1, &late)) goto timeout;
  {
    // the entry counted into its cell
    int slot = 1;
    if (on) slot = -1 - atomicSub(&cellmap[key], 1);
    if (on && s == 0 && err) atomicMin(&ctl[kErr], (m + 1) * 4 + err);
    if (!couple_barrier(arrived, 2, &late)) goto timeout;
    // k_ibm_claim's work
    const bool won = on && slot == 0;
    const int n0 = won ? -1 - xload(&cellmap[key]) : 0;
    const unsigned long long mask = __ballot(won);
    int upto = n0;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(upto, off, 64);
      if (s >= off) upto += o;
    }
    {
      const unsigned ny = a.st.nd[1], nz = a.st.nd[2], plane = ny * nz;
      const unsigned x = key / plane, r = key - x * plane, y = r / nz;
      const int v[3] = {(int)x, (int)y, (int)(r - y * nz)};
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        int lo = won ? v[k] : 0x7fffffff, hi = won ? v[k] : -1;
        for (int off = 32; off > 0; off >>= 1) {
          lo = min(lo, __shfl_xor(lo, off, 64));
          hi = max(hi, __shfl_xor(hi, off, 64));
        }
        if (s == 0) {
          wbox[w][k] = lo;
          wbox[w][3 + k] = hi;
        }
      }
    }
    if (s == 63) {
      wave_won[w] = __popcll(mask);
      wave_ent[w] = upto;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      int nw = 0, ne = 0;
      for (int k = 0; k < NW; ++k) {
        nw += wave_won[k];
        ne += wave_ent[k];
      }
      blk_base = nw ? atomicAdd(reinterpret_cast<unsigned long long *>(&ctl[kNew]),
                                ((unsigned long long)ne << 32) | (unsigned long long)nw)
                    : 0ULL;
    }
    if (threadIdx.x >= 64 && threadIdx.x < 70) {
      const int k = threadIdx.x - 64;
      int r = wbox[0][k];
      for (int q = 1; q < NW; ++q) r = k < 3 ? min(r, wbox[q][k]) : max(r, wbox[q][k]);
      if (k < 3) atomicMin(&ctl[kBoxLo + k], r);
      else atomicMax(&ctl[kBoxLo + k], r);
    }
    __syncthreads();
    if (won) {
      int b = (int)(blk_base & 0xffffffffULL) + __popcll(mask & ((1ULL << s) - 1ULL));
      int p = (int)(blk_base >> 32) + upto - n0;
      for (int k = 0; k < w; ++k) {
        b += wave_won[k];
        p += wave_ent[k];
      }
      a.cell[b] = (long long)key;
      xstore(&a.ptr[b], p);
      atomicExch(&cellmap[key], b);
    }
    if (!couple_barrier(arrived, 3, &late)) goto timeout;
    // k_ibm_fill's and k_ibm_rank's work
    const int nband = xload(&ctl[kNew]);
    int b = xload(&cellmap[key]);
    bool placed = b >= 0 && b < nband;
    if (!placed) b = 0;
    const int p0 = xload(&a.ptr[b]), n = placed ? (b + 1 < nband ? xload(&a.ptr[b + 1]) : E) - p0 : 0;
    placed = placed && (!on || (slot >= 0 && slot < n));
    if (!placed) atomicMin(&ctl[kErr], 4);
    if (first) {
      ctl[kNband] = nband;
      a.ptr[nband] = E;
    }
    if (on && placed) xstore(&a.tmp[p0 + slot], e);
    for (int i = threadIdx.x; i < 12 * M; i += kCoupleThreads) lds.W[0][i] = xload(&a.st.Ew[i]);
    if (!couple_barrier(arrived, 4, &late)) goto timeout;
    int rank = 0, near[B];
#pragma unroll
    for (int j = 0; j < B; ++j) near[j] = j < n ? xload(&a.tmp[p0 + j]) : 0x7fffffff;
#pragma unroll
    for (int j = 0; j < B; ++j) rank += near[j] < e ? 1 : 0;
    for (int j0 = B; j0 < n; j0 += 16) {
      int v[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) v[j] = xload(&a.tmp[p0 + min(j0 + j, n - 1)]);
#pragma unroll
      for (int j = 0; j < 16; ++j) rank += j0 + j < n && v[j] < e ? 1 : 0;
    }
    if (on && placed && rank < n) {
      const unsigned long long *q = reinterpret_cast<const unsigned long long *>(&a.went[p0 + rank]);
      unsigned long long *o = const_cast<unsigned long long *>(q);
      xstore(&o[0], ((unsigned long long)__float_as_uint(fwy) << 32) | __float_as_uint(fwx));
      xstore(&o[1], ((unsigned long long)(unsigned)m << 32) | __float_as_uint(fwz));
    }
    // the cell's list: its entries in order, from the placed ones where all are
    // in registers, else from the list itself once every workgroup has written
    // its part (plain reads from then on)
    const float4 *we = a.went + p0;
    float4 q[B];
    couple_arrive(&ctl[kListed]);
    if (__syncthreads_or(n > B)) {
      if (!couple_wait(&ctl[kListed], 1, &late)) goto timeout;
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
#pragma unroll
      for (int j = 0; j < B; ++j) {
        q[j] = we[max(min(j, n - 1), 0)];
        q[j].w = __int_as_float((int)min((unsigned)__float_as_int(q[j].w), (unsigned)(M - 1)));
      }
    } else {
      sort16(near);
#pragma unroll
      for (int j = 0; j < B; ++j) {
        const int x = j < n ? (int)min((unsigned)near[j], (unsigned)(E - 1)) : 0, k = x >> 6;
        q[j] = make_float4(lds.W[k][(x >> 4) & 3], lds.W[k][4 + ((x >> 2) & 3)], lds.W[k][8 + (x & 3)],
                           __int_as_float(k));
      }
    }
    // (past the list's end: a zero value with zero weights, u - 0 = u)
#pragma unroll
    for (int j = 0; j < B; ++j)
      if (j >= n) q[j] = make_float4(0.0f, 0.0f, 0.0f, __int_as_float(M));
    __syncthreads();  // (the weights' LDS is the rounds' from here on)
    if (threadIdx.x < 4) fx[threadIdx.x][M] = 0.0;

    // the forcing rounds
    const double rx = (double)fwx, ry = (double)fwy, rz = (double)fwz;
    double ef = 0.0, u1 = u[0], u2 = u[1], u3 = u[2];
    const int nmax = [&] {
      int v = n;
      for (int off = 32; off > 0; off >>= 1) v = max(v, __shfl_xor(v, off, 64));
      return __builtin_amdgcn_readfirstlane(v);
    }();
    for (int r = 0;; ++r) {
      t[w][0][s] = ((u1 * rx) * ry) * rz;
      t[w][1][s] = ((u2 * rx) * ry) * rz;
      t[w][2][s] = ((u3 * rx) * ry) * rz;
      wave_sync();
      double *xo = a.xch + (long long)(r & 1) * 4 * M;
      {
        double v = 0.0, x[2][16];
#pragma unroll
        for (int k = 0; k < 16; ++k) x[0][k] = t[w][c][k];
#pragma unroll
        for (int g = 0; g < 4; ++g) {  // (sixteen terms read ahead of those added)
          if (g < 3) {
#pragma unroll
            for (int k = 0; k < 16; ++k) x[(g + 1) & 1][k] = t[w][c][16 * (g + 1) + k];
          }
#pragma unroll
          for (int k = 0; k < 16; ++k) v = v + x[g & 1][k];
        }
        const double d = ev - v, F = d * am;
        ef = ef + F;
        const double d0 = lane_value(d, 0), d1 = lane_value(d, 1), d2 = lane_value(d, 2);
        if (on && s < 4) xstore(&xo[(long long)s * M + m], s < 3 ? F * a.invh3 : (fabs(d0) + fabs(d1)) + fabs(d2));
      }
      if (!couple_barrier(arrived, 5 + r, &late)) goto timeout;
      for (int i = threadIdx.x; i < M; i += kCoupleThreads) {
        double v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = xload(&xo[(long long)k * M + i]);
#pragma unroll
        for (int k = 0; k < 4; ++k) fx[k][i] = v[k];
      }
      __syncthreads();
      // the residual, in mdf_tl_sum's order (256 strided sums, wave trees, the four in order)
      {
        double p = 0.0;
        for (int i = threadIdx.x; i < M; i += 256) p = p + fx[3][i];
        p = wave_sum(p);
        if (s == 0) part[w] = p;
      }
      // the correction of this lane's cell, its entries in order
#pragma unroll
      for (int h = 0; h < B; h += 8) {
        if (h >= nmax) break;
        double f[8][3];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          int k = __float_as_int(q[h + j].w);
          asm volatile("" : "+v"(k));  // (no addresses kept across the rounds)
          f[j][0] = fx[0][k]; f[j][1] = fx[1][k]; f[j][2] = fx[2][k];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const double qx = (double)q[h + j].x, qy = (double)q[h + j].y, qz = (double)q[h + j].z;
          u1 = u1 - ((f[j][0] * qx) * qy) * qz;
          u2 = u2 - ((f[j][1] * qx) * qy) * qz;
          u3 = u3 - ((f[j][2] * qx) * qy) * qz;
        }
      }
      for (int j0 = B; j0 < n; j0 += 8) {
        float4 g[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) g[j] = we[min(j0 + j, n - 1)];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int k = (int)min((unsigned)__float_as_int(g[j].w), (unsigned)(M - 1));
          const double qx = (double)g[j].x, qy = (double)g[j].y, qz = (double)g[j].z;
          const double x1 = ((fx[0][k] * qx) * qy) * qz, x2 = ((fx[1][k] * qx) * qy) * qz,
                       x3 = ((fx[2][k] * qx) * qy) * qz;
          u1 = j0 + j < n ? u1 - x1 : u1;
          u2 = j0 + j < n ? u2 - x2 : u2;
          u3 = j0 + j < n ? u3 - x3 : u3;
        }
      }
      __syncthreads();
      double tol = 0.0;
      for (int k = 0; k < 4; ++k) tol = tol + part[k];
      if (first) mdf_decide(ctl, a.mt.dstate, tol, a.mt.dsum, a.mt.Uref, a.mt.ntol, a.mt.dtol, a.mt.skip,
                            MdfWords{r, 0, 0, ref});
      // (mdf_decide's condition without a learned guess, after r + 1 iterations)
      if (!isfinite(tol) || !(r + 1 < a.mt.ntol && tol / (a.mt.dsum * a.mt.Uref) > a.mt.dtol)) {
        if (first) ctl[kRan] = r;
        break;
      }
    }
    if (on && s < 3) a.Eforce[3LL * m + s] = ef;
    if (on && placed && rank == 0) {  // the cell's first entry
      a.ma.band_u[b] = u1;
      a.ma.band_u[a.ma.cap + b] = u2;
      a.ma.band_u[2LL * a.ma.cap + b] = u3;
    }
    return;
  }
timeout:
  if (threadIdx.x == 0) atomicMin(&ctl[kErr], 2);
}

// The control words and the last residual of a coupling call, written into
// pinned host memory (read by the host after the stream's synchronisation).
struct IbmReport {
  int ctl[kCtlWords];
  double dmax;
};

// The end of a coupling call in one launch: the beam loads, the spreading and
// the report.
// Beam nodal loads lodFlow (Solidbody.f90:944-967): per degree of freedom, the
// sum over its markers in marker order of 0.5*F (translational) or
// 0.5*(r x F) (rotational) with r the arm from the element axis midpoint;
// dof_list entry: marker id, dof_kind[d] = component (0..2 force, 3..5
// moment).  The leading dof_blocks workgroups form them with one wave per
// degree of freedom: the lanes form the DOF's terms into LDS, then lane 0 adds
// them in list order.
// Eulerian force of every band cell (ResetVolumeForce_ FluidDomain.f90:
// 1195-1206, FluidVolumeForce_ Solidbody.f90:968-977, add_volume_force_
// FluidDomain.f90:1182-1193): (0 - sum F/h^3*rx*ry*rz) + VF, by the other
// band_blocks workgroups (band_cells_reduce, workgroup blk of them), the first of which copies the
// control words into the report (the last k_correct has made the stop test,
// so they are final).
constexpr int kLoadChunk = 256;

struct IbmFinishArgs {
  int *ctl;
  const double *dstate;
  IbmReport *rep;
  int cap;
  const int *ptr;
  const float4 *went;
  const double *Eforce;
  double invh3, VF1, VF2, VF3;
  double *band_F;
  int ndof, dof_blocks, band_blocks, pass_cap;
  const int *dof_ptr, *dof_list, *dof_elem, *dof_kind, *marker_elem;
  const double *elem_xc, *Exyz;
  double *lod;
};

__device__ __forceinline__ double load_term(const IbmFinishArgs &a, int kind, int m, int el) {
  if (kind < 3) return 0.5 * a.Eforce[3LL * m + kind];
  const double r1 = a.Exyz[3LL * m] - a.elem_xc[3LL * el];
  const double r2 = a.Exyz[3LL * m + 1] - a.elem_xc[3LL * el + 1];
  const double r3 = a.Exyz[3LL * m + 2] - a.elem_xc[3LL * el + 2];
  const double F1 = a.Eforce[3LL * m], F2 = a.Eforce[3LL * m + 1], F3 = a.Eforce[3LL * m + 2];
  double val;
  if (kind == 3) val = r2 * F3 - r3 * F2;
  else if (kind == 4) val = r3 * F1 - r1 * F3;
  else val = r1 * F2 - r2 * F1;
  return 0.5 * val;
}

__global__ __launch_bounds__(256) void k_ibm_finish(IbmFinishArgs a) {
  if ((int)blockIdx.x < a.dof_blocks) {
    __shared__ double term[4][kLoadChunk];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int d = blockIdx.x * 4 + w;
    if (d >= a.ndof) return;  // whole waves; no workgroup barrier follows
    const int kind = a.dof_kind[d];
    const int j0 = a.dof_ptr[d], j1 = a.dof_ptr[d + 1];
    double acc = 0.0;
    for (int base = j0; base < j1; base += kLoadChunk) {
      const int n = min(kLoadChunk, j1 - base);
      for (int q = lane; q < n; q += 64) term[w][q] = load_term(a, kind, a.dof_list[base + q], a.dof_elem[base + q]);
      wave_sync();
      if (lane == 0)
        for (int q = 0; q < n; ++q) acc = acc + term[w][q];
      wave_sync();
    }
    if (lane == 0) a.lod[d] = acc;
    return;
  }
  const int blk = (int)blockIdx.x - a.dof_blocks;
  if (blk == 0 && threadIdx.x < kCtlWords) a.rep->ctl[threadIdx.x] = a.ctl[threadIdx.x];
  if (blk == 0 && threadIdx.x == 0) a.ctl[kArrived] = a.ctl[kListed] = 0;
  if (blk == 0 && threadIdx.x == 0) a.rep->dmax = a.dstate[0];
  if (band_build_failed(a.ctl[kErr])) {  // (uniform) the band is left empty
    if (blk == 0 && threadIdx.x <= kNband)
      a.ctl[threadIdx.x] = threadIdx.x < 3 ? 0x7fffffff : (threadIdx.x < 6 ? -1 : 0);
    return;
  }
  band_cells_reduce<true>(blk, a.ctl[kNband], a.band_blocks, a.cap, a.ptr, a.went, a.Eforce, a.invh3, a.band_F,
                          a.VF1, a.VF2, a.VF3, a.pass_cap);
}

// ---------------------------------------------------------------------------
// Learned warm start (no counterpart in the reference)
//
// The forcing loop is linear in the accumulated marker force: after j rounds
// from the zero guess, Eforce = E_j and the band velocity is
// u0 - S(E_j h^-3 / (2 rho)) with S the spreading of the stencil weights.  A
// guess of E_k applied as one correction of the uncorrected band velocity u0
// therefore puts the loop in the state of round k, and the loop goes on from
// iteration k + 1 to the same cap and tolerance.  The network predicts E_k
// as a correction to the marker's force of the previous call:
//   E_k ~ Eprev + Uref |Ea| net(X)
// and is trained on E_k recorded from plain calls.

// Features of every marker for the network, one wave per marker: the
// interpolated velocity of the uncorrected band (as k_interp forms it), the
// marker velocity, the marker's force of the previous call and its normal:
//   X = [U/Uref, V/Uref, Fprev/(Uref |Ea|), n]
__global__ __launch_bounds__(256) void k_ws_features(int M, const int *__restrict__ bidx,
                                                     const float *__restrict__ Ew,
                                                     const double *__restrict__ band_u, int cap,
                                                     const double *__restrict__ Evel,
                                                     const double *__restrict__ Ea,
                                                     const double *__restrict__ Eprev,
                                                     const double *__restrict__ Enrm, double Uref,
                                                     float *__restrict__ X) {
  __shared__ double t[4][3][64];
  const int w = threadIdx.x >> 6, s = threadIdx.x & 63;
  const int m = blockIdx.x * 4 + w;
  if (m < M) {
    const int b = bidx[64LL * m + s];
    const float *W = Ew + 12LL * m;
    const double rx = (double)W[s >> 4], ry = (double)W[4 + ((s >> 2) & 3)], rz = (double)W[8 + (s & 3)];
    t[w][0][s] = ((band_u[b] * rx) * ry) * rz;
    t[w][1][s] = ((band_u[cap + b] * rx) * ry) * rz;
    t[w][2][s] = ((band_u[2LL * cap + b] * rx) * ry) * rz;
  }
  __syncthreads();
  if (m < M && s == 0) {
    double v[3] = {0.0, 0.0, 0.0};
    for (int k = 0; k < 64; ++k) {
      v[0] = v[0] + t[w][0][k];
      v[1] = v[1] + t[w][1][k];
      v[2] = v[2] + t[w][2][k];
    }
    const double fs = Uref * fabs(Ea[m]);
    float *x = X + 12LL * m;
    for (int c = 0; c < 3; ++c) {
      x[c] = (float)(v[c] / Uref);
      x[3 + c] = (float)(Evel[3LL * m + c] / Uref);
      x[6 + c] = (float)(fs > 0.0 ? Eprev[3LL * m + c] / fs : 0.0);
      x[9 + c] = Enrm ? (float)Enrm[3LL * m + c] : 0.f;
    }
  }
}

// the network's guess of E_k as the starting force: Eforce = Eprev + Y Uref
// |Ea|, fT = Eforce * invh3 (applied to the band by k_correct as one
// correction of the uncorrected velocity)
__global__ __launch_bounds__(256) void k_ws_apply(int M, const float *__restrict__ Y, const double *__restrict__ Ea,
                                                  const double *__restrict__ Eprev, double Uref, double invh3,
                                                  double *__restrict__ Eforce, double *__restrict__ fT) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 3 * M) return;
  const double F0 = Eprev[i] + (double)Y[i] * (Uref * fabs(Ea[i / 3]));
  Eforce[i] = F0;
  fT[i] = F0 * invh3;
}

// restart from the zero guess when the stop test asked for it
__global__ __launch_bounds__(256) void k_ws_fallback(int M, int *__restrict__ ctl, double *__restrict__ Eforce) {
  if (ctl[kFallback] != 1) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 3 * M) Eforce[i] = 0.0;
}
__global__ void k_ws_fallback_end(int *__restrict__ ctl) {
  if (threadIdx.x == 0 && ctl[kFallback] == 1) ctl[kFallback] = 2;
}

// training target of a plain call, (E_k - Eprev) / (Uref |Ea|) with E_k the
// force after `skip` rounds (the final force when the loop stopped earlier),
// then Eprev = the call's final force, the previous force of the next call
__global__ __launch_bounds__(256) void k_ws_targets(int M, const int *__restrict__ ctl, int skip,
                                                    const double *__restrict__ Eforce,
                                                    const double *__restrict__ Esnap,
                                                    const double *__restrict__ Ea, double Uref, int record,
                                                    float *__restrict__ Y, double *__restrict__ Eprev) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 3 * M) return;
  if (record) {
    const double fs = Uref * fabs(Ea[i / 3]);
    const double Ek = (skip > 0 && ctl[kIters] >= skip) ? Esnap[i] : Eforce[i];
    Y[i] = (float)(fs > 0.0 ? (Ek - Eprev[i]) / fs : 0.0);
  }
  Eprev[i] = Eforce[i];
}

}  // namespace fsil
