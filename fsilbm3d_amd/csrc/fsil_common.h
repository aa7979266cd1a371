// Shared definitions of the FSILBM3D MI355X hot-path library (device + host).
#pragma once
#include <hip/hip_runtime.h>
#include <cstddef>
#include <cstdint>

namespace fsil {

constexpr int Q = 19;

// barrier of the lanes of one wave (they run in lockstep; the fences keep the
// compiler from moving LDS accesses across it)
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// D3Q19 lattice, in the reference's direction order (ConstParams.f90:11-25).
__host__ __device__ constexpr int ex(int q) {
  constexpr int e[Q] = {0, 1, -1, 0, 0, 0, 0, 1, -1, 1, -1, 1, -1, 1, -1, 0, 0, 0, 0};
  return e[q];
}
__host__ __device__ constexpr int ey(int q) {
  constexpr int e[Q] = {0, 0, 0, 1, -1, 0, 0, 1, 1, -1, -1, 0, 0, 0, 0, 1, -1, 1, -1};
  return e[q];
}
__host__ __device__ constexpr int ez(int q) {
  constexpr int e[Q] = {0, 0, 0, 0, 0, 1, -1, 0, 0, 0, 0, 1, 1, -1, -1, 1, 1, -1, -1};
  return e[q];
}
__host__ __device__ constexpr int oppo(int q) {
  constexpr int o[Q] = {0, 2, 1, 4, 3, 6, 5, 10, 9, 8, 7, 14, 13, 12, 11, 18, 17, 16, 15};
  return o[q];
}
// weights 1/3, 1/18 (axis), 1/36 (diagonal), each the correctly rounded double
__host__ __device__ constexpr double wt(int q) {
  return q == 0 ? 1.0 / 3.0 : (q <= 6 ? 1.0 / 18.0 : 1.0 / 36.0);
}

// Population planes in global memory.  A uniform plane base is kept in scalar
// registers (the empty asm stops the compiler from folding it back into
// per-lane 64-bit address arithmetic), so every access is one scalar base plus
// a 32-bit per-lane byte offset, and the base advances by one plane per
// direction with two scalar adds.
template <typename T> using gptr = __attribute__((address_space(1))) T *;
template <typename T>
__device__ __forceinline__ gptr<T> sbase(gptr<T> g) {
  asm volatile("" : "+s"(g));
  return g;
}

// a 32-bit per-lane offset defined afresh where it is used, so the address
// selection there sees its zero extension (scalar base + 32-bit offset form)
__device__ __forceinline__ unsigned voff(unsigned o) {
  asm volatile("" : "+v"(o));
  return o;
}

// s + row . v in ascending order, row = 19 launch-uniform values read through
// scalar registers.  The empty asm makes the row's reads wait for `after`, the
// result of an earlier row: hoisted to the front of an unrolled 19 x 19
// product the reads take more registers than there are (the kernels spilled
// 160-1700 of them).  FP64 MRT with a volume force, 160x96x77 cells: 332 us
// per launch with the spills, 123 us this way (its 2,900 FP64 operations per
// cell take about 55 us, its 304 bytes 57 us).
template <typename T> using cptr = __attribute__((address_space(4))) const T *;
template <bool FMA, typename T>
__device__ __forceinline__ T row_dot(const T *row, const T (&v)[Q], T s, T after) {
  cptr<T> c = (cptr<T>)row;
  asm volatile("" : "+s"(c) : "v"(after));
#pragma unroll
  for (int j = 0; j < Q; ++j) {
    if constexpr (FMA) s = __builtin_fmaf(c[j], v[j], s);
    else s = s + c[j] * v[j];
  }
  return s;
}

// The 19 values of one cell, v[q] = plane q at byte offset off.  nt streams
// them past the caches (nontemporal); the choice is uniform over a launch.
template <typename T>
__device__ __forceinline__ void load_cell(T (&v)[Q], const T *planes, size_t plane_bytes, unsigned off, bool nt) {
  gptr<const char> base = sbase((gptr<const char>)planes);
  if (nt) {
    const unsigned o = voff(off);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      v[q] = __builtin_nontemporal_load((gptr<const T>)(base + o));
      base = sbase(base + plane_bytes);
    }
  } else {
    const unsigned o = voff(off);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      v[q] = *((gptr<const T>)(base + o));
      base = sbase(base + plane_bytes);
    }
  }
}

// Boundary codes (ConstParams.f90:31-34)
enum BcCode {
  BC_FLUID = 0,
  BC_FLUID_FATHER = 1,
  BC_EQ_DIRICHLET = 101,
  BC_NEQ_DIRICHLET = 102,
  BC_EXTRAP1 = 103,
  BC_EXTRAP2 = 104,
  BC_WALL = 201,
  BC_MOVING_WALL = 202,
  BC_WALL_HALFWAY = 203,
  BC_MOVING_WALL_HALFWAY = 204,
  BC_PERIODIC = 301,
  BC_SYMMETRIC = 302,
};

// Push of one cell's post-collision values: v[q] to plane q at cell
// n + step_x + step_y + step_z, where the steps are st[0..5] = (+x, -x, +y,
// -y, +z, -z) for the axes e_q moves along (periodic wrap folded into them).
// The destinations are formed inside each branch, next to their stores.
template <typename T>
__device__ __forceinline__ unsigned push_offset(int q, unsigned n, const unsigned (&st)[6]) {
  const unsigned sx = ex(q) > 0 ? st[0] : (ex(q) < 0 ? st[1] : 0u);
  const unsigned sy = ey(q) > 0 ? st[2] : (ey(q) < 0 ? st[3] : 0u);
  const unsigned sz = ez(q) > 0 ? st[4] : (ez(q) < 0 ? st[5] : 0u);
  return (n + sx + sy + sz) * (unsigned)sizeof(T);
}

template <typename T>
__device__ __forceinline__ void store_cell(const T (&v)[Q], T *planes, size_t plane_bytes, unsigned n,
                                           const unsigned (&st)[6], bool nt) {
  gptr<char> base = sbase((gptr<char>)planes);
  if (nt) {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      __builtin_nontemporal_store(v[q], (gptr<T>)(base + push_offset<T>(q, n, st)));
      base = sbase(base + plane_bytes);
    }
  } else {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      *((gptr<T>)(base + push_offset<T>(q, n, st))) = v[q];
      base = sbase(base + plane_bytes);
    }
  }
}

// The z faces that a collide launch applies itself (whole-row workgroups):
// their codes (0: none) and the active x and y faces, whose nodes (the rim)
// k_rim completes after the launch.
struct ZFaces {
  int code[2];  // z-, z+: BC_SYMMETRIC, BC_WALL, BC_WALL_HALFWAY or 0
  int rim;      // bit k: face k (x-, x+, y-, y+) is active
  __host__ __device__ bool any() const { return code[0] != 0 || code[1] != 0; }
  __host__ __device__ bool walls() const {
    return (code[0] != 0 && code[0] != BC_SYMMETRIC) || (code[1] != 0 && code[1] != BC_SYMMETRIC);
  }
  __host__ __device__ bool halfway() const { return code[0] == BC_WALL_HALFWAY || code[1] == BC_WALL_HALFWAY; }
  // whether the nodes of a row's x (y) neighbours e = -1, 0, 1, periodic, are on an active x (y) face: r[e + 1]
  __device__ __forceinline__ void rims(int x, int y, int xd, int yd, bool (&rx)[3], bool (&ry)[3]) const {
#pragma unroll
    for (int e = -1; e <= 1; ++e) {
      const int xx = x + e < 0 ? xd - 1 : (x + e == xd ? 0 : x + e), yy = y + e < 0 ? yd - 1 : (y + e == yd ? 0 : y + e);
      rx[e + 1] = (xx == 0 && (rim & 1)) || (xx == xd - 1 && (rim & 2));
      ry[e + 1] = (yy == 0 && (rim & 4)) || (yy == yd - 1 && (rim & 8));
    }
  }
};

__host__ __device__ constexpr int mirror_z(int q) {
  for (int p = 0; p < Q; ++p)
    if (ex(p) == ex(q) && ey(p) == ey(q) && ez(p) == -ez(q)) return p;
  return q;
}

// Rows that end on z faces, in whole-row workgroups.  v holds the exchanged
// values (those that arrive at the thread's own z).  Where the face sets an
// incoming population q of a node from one that arrives there too, this thread
// has it: the mirrored one goes to q's own destination, the opposite one to
// the node on the other side, the halfway wall's (hw: at the ends of a row the
// thread's five populations that move into the face, before the exchange,
// ascending directions) to the thread's own cell.  Rim nodes get the plain
// streamed values instead, as k_rim expects them.
// As launches of their own the z faces touched a cache line per population
// and node: 57 us for the 147,456 nodes of 384x192x192 FP64 beside 790 for the
// collision, 302 for 1024x384x384 FP32.
//
// Symmetry alone replaces values in place, and the plain stores follow.
template <typename T>
__device__ __forceinline__ void mirror_faces(T (&v)[Q], const ZFaces &zf, int x, int y, int z, int xd, int yd,
                                             int zd) {
  if (z != 0 && z != zd - 1) return;
  bool rx[3], ry[3];
  zf.rims(x, y, xd, yd, rx, ry);
  const bool lo = z == 0 && zf.code[0] != 0, hi = z != 0 && zf.code[1] != 0;
#pragma unroll
  for (int q = 0; q < Q; ++q)
    if (ez(q) > 0) {
      const bool plain = rx[ex(q) + 1] || ry[ey(q) + 1];
      const T up = v[q], down = v[mirror_z(q)];
      if (lo && !plain) v[q] = down;
      if (hi && !plain) v[mirror_z(q)] = up;
    }
}

// Walls store to other rows too.
template <typename T>
__device__ __forceinline__ void store_cell_faces(const T (&v)[Q], const T (&hw)[5], T *planes, size_t plane_bytes,
                                                 unsigned n, const unsigned (&st)[6], bool nt, const ZFaces &zf,
                                                 int x, int y, int z, int xd, int yd, int zd) {
  gptr<char> base = sbase((gptr<char>)planes);
  auto put = [&](T val, unsigned off) {
    if (nt) __builtin_nontemporal_store(val, (gptr<T>)(base + off));
    else *((gptr<T>)(base + off)) = val;
  };
  bool rx[3], ry[3];
  zf.rims(x, y, xd, yd, rx, ry);
  const int code = z == 0 ? zf.code[0] : (z == zd - 1 ? zf.code[1] : 0);
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    T val = v[q];
    unsigned off = push_offset<T>(q, n, st);
    bool put1 = true;
    if (ez(q) != 0) {
      const bool in = code != 0 && (ez(q) > 0 ? z == 0 : z == zd - 1);  // q comes out of this thread's face
      if (in) {
        const bool to_rim = rx[ex(q) + 1] || ry[ey(q) + 1];
        if (code == BC_SYMMETRIC) {
          if (!to_rim) val = v[mirror_z(q)];
        } else {
          const bool wall = code == BC_WALL;
          const bool set = wall ? !(rx[1 - ex(q)] || ry[1 - ey(q)]) : !(rx[1] || ry[1]);
          if (set) {
            if (to_rim) put(val, off);
            // the five populations of one z direction in ascending order: 5 11 12 15 16 and 6 13 14 17 18
            constexpr int pos[Q] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 1, 2, 1, 2, 3, 4, 3, 4};
            val = wall ? v[oppo(q)] : hw[pos[oppo(q)]];
            off = wall ? push_offset<T>(oppo(q), n, st) : n * (unsigned)sizeof(T);
          } else {
            put1 = to_rim;
          }
        }
      }
    }
    if (put1) put(val, off);
    base = sbase(base + plane_bytes);
  }
}

// the populations of hw in store_cell_faces: those a thread at z = 0 (z = zd-1)
// moves into its face
template <typename T>
__device__ __forceinline__ void face_bound(T (&hw)[5], const T (&post)[Q], int z) {
  int k = 0, l = 0;
#pragma unroll
  for (int q = 0; q < Q; ++q)
    if (ez(q) < 0) {
      hw[k] = post[q];
      ++k;
    }
  if (z != 0) {
#pragma unroll
    for (int q = 0; q < Q; ++q)
      if (ez(q) > 0) {
        hw[l] = post[q];
        ++l;
      }
  }
}

// Whole z-rows per workgroup (blockDim.x == zDim; every thread takes part):
// the ten values that move along z (e_z = +-1) are exchanged
// through LDS so that each thread stores, at its own z, the value arriving
// there from z - e_z (periodic within the row).  A wave's stores then cover
// whole cache lines instead of lines shifted by one value.  lds holds
// 10 * blockDim.x * blockDim.y values.
template <typename T>
__device__ __forceinline__ void shift_rows_z(T (&post)[Q], T *lds) {
  const int nt = (int)(blockDim.x * blockDim.y);
  const int zr = (int)threadIdx.x, zd = (int)blockDim.x, row = (int)threadIdx.y * zd;
  const int t = row + zr;
  int k = 0;
#pragma unroll
  for (int q = 0; q < Q; ++q)
    if (ez(q) != 0) lds[(k++) * nt + t] = post[q];
  __syncthreads();
  const int from_m = row + (zr == 0 ? zd - 1 : zr - 1);  // sender of e_z = +1
  const int from_p = row + (zr == zd - 1 ? 0 : zr + 1);  // sender of e_z = -1
  k = 0;
#pragma unroll
  for (int q = 0; q < Q; ++q)
    if (ez(q) != 0) post[q] = lds[(k++) * nt + (ez(q) > 0 ? from_m : from_p)];
}

// The same exchange for rows of whole waves (blockDim.x a multiple of 64):
// inside a wave the values move by lane permutes (no LDS allocation); only
// each wave's first and last lanes go through edge[], 20 values per wave
// (80 bytes per wave for FP32).  Leaves the LDS free for a large workgroup
// that shares the CU.
__device__ __forceinline__ void shift_rows_z_waves(float (&post)[Q], float *edge) {
  const int zd = (int)blockDim.x, wpr = zd >> 6;
  const int lane = (int)threadIdx.x & 63, wr = (int)threadIdx.x >> 6;
  const int w = (int)threadIdx.y * wpr + wr, rw0 = w - wr;
  if (lane == 0 || lane == 63) {
    int k = 0;
#pragma unroll
    for (int q = 0; q < Q; ++q)
      if (ez(q) != 0) edge[(w * 2 + (lane == 63 ? 1 : 0)) * 10 + (k++)] = post[q];
  }
  __syncthreads();
  const int prev_w = rw0 + (wr == 0 ? wpr - 1 : wr - 1), next_w = rw0 + (wr == wpr - 1 ? 0 : wr + 1);
  const int src_m = (lane == 0 ? 0 : lane - 1) << 2, src_p = (lane == 63 ? 63 : lane + 1) << 2;
  int k = 0;
#pragma unroll
  for (int q = 0; q < Q; ++q)
    if (ez(q) != 0) {
      const int v = __builtin_amdgcn_ds_bpermute(ez(q) > 0 ? src_m : src_p, __float_as_int(post[q]));
      float f = __int_as_float(v);
      if (ez(q) > 0 && lane == 0) f = edge[(prev_w * 2 + 1) * 10 + k];
      if (ez(q) < 0 && lane == 63) f = edge[(next_w * 2 + 0) * 10 + k];
      post[q] = f;
      ++k;
    }
}

}  // namespace fsil
