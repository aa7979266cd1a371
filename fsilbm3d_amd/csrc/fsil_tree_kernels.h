// Father/son (refinement ratio 2) halo exchange of the block tree, FP64
// plain form (gaoak/FSILBM3D src/LBMBlockComm.f90).
//
// A pair keeps, for every son face whose boundary code is BCfluid (0), two
// copies of the father plane under it: level 1 (taken before the father's
// collision) and level 2 (after its boundary faces).  Planes are stored
// [q][a][b] with b the fast in-plane index (z for x and y faces, y for z
// faces), as the reference's fIn_F*t* arrays (LBMBlockComm.f90:201-245).
//
// The reference builds each fine plane in passes over a scratch array
// (interpolate_fIn, LBMBlockComm.f90:808-914); here each son node forms the
// passes' sums from the coarse plane, in the same association order, so every
// value is the one the passes produce.
#pragma once
#include "fsil_lbm_kernels.h"

namespace fsil {

struct TreeFace {
  int active;       // sds != 0
  int fixedF;       // father coordinate (0-based) of the plane along the face axis
  int fixedS;       // son coordinate (0-based) of the son boundary plane
  int fixedFi;      // father coordinate of the first inner father plane (son-to-father)
  int fixedSi;      // son coordinate of the son layer delivered to the father
  int aF, bF;       // coarse plane extent
  int aS, bS;       // son plane extent
  long long off;    // offset of the level-1 plane in the pair buffer; level 2 follows
};

struct TreeArgs {
  double *__restrict__ ff;  // father state (current buffer)
  double *__restrict__ fs;  // son state (current buffer)
  double *__restrict__ planes;
  int fxd, fyd, fzd;
  long long fN;
  int sxd, syd, szd;
  long long sN;
  int f0[3];        // father start (0-based) of the plane window, per axis
  int si0[3];       // son inner-layer start (0-based), per axis (son-to-father)
  int sicnt[3];     // number of delivered son nodes per axis (step 2)
  int fi0[3];       // father inner start (0-based), per axis
  TreeFace face[6];
  double coeff;     // grid-transform coefficient of this launch
  double hv[3];     // 0.5*VF*dh of the block whose VF the transform uses
};

// The exchange kernels take one thread per (node, direction), kTreeNodes nodes
// per workgroup of kTreeNodes x 19 threads, threadIdx.y the direction: every
// thread brings its population into LDS and, for the rescaling, forms the
// node's moments from there itself.  Bound: latency (a son face holds a few
// thousand nodes).  One thread per node, walking the 19 directions' sixteen
// reads one after the other, took 92.7 us per father-to-son transfer of a
// 65x49x49 son (16,706 face nodes) and 12.7 us per delivery, against 10.9 and
// 4.9 this way.
constexpr int kTreeNodes = 32;

// fIn_GridTransform (LBMBlockComm.f90:958-979): Dupuis-Chopard rescaling of
// the non-equilibrium part of population q by coeff, equilibrium from the
// node's own moments (f: its 19 populations).
__device__ __forceinline__ double grid_transform(int q, const double (&f)[Q], double coeff, const double (&hv)[3]) {
  double rho, m1, m2, m3;
  moments(f, rho, m1, m2, m3);
  const double u1 = (m1 + hv[0]) / rho;
  const double u2 = (m2 + hv[1]) / rho;
  const double u3 = (m3 + hv[2]) / rho;
  const double uSqr = (u1 * u1 + u2 * u2) + u3 * u3;
  const double base = 1.0 - 1.5 * uSqr;
  switch (q) {
#define FSIL_GT(k)                                                          \
  case k: {                                                                 \
    const double ux = dotu<k>(u1, u2, u3);                                  \
    const double feq = (wt(k) * rho) * (base + ux * (3.0 + 4.5 * ux));    \
    return feq + coeff * (f[k] - feq);                                      \
  }
    FSIL_GT(0) FSIL_GT(1) FSIL_GT(2) FSIL_GT(3) FSIL_GT(4) FSIL_GT(5) FSIL_GT(6)
    FSIL_GT(7) FSIL_GT(8) FSIL_GT(9) FSIL_GT(10) FSIL_GT(11) FSIL_GT(12) FSIL_GT(13)
    FSIL_GT(14) FSIL_GT(15) FSIL_GT(16) FSIL_GT(17) FSIL_GT(18)
#undef FSIL_GT
  }
  return 0.0;
}

// the node's populations from LDS ([direction][node])
__device__ __forceinline__ void tree_node(double (&f)[Q], const double (*sh)[kTreeNodes]) {
#pragma unroll
  for (int q = 0; q < Q; ++q) f[q] = sh[q][threadIdx.x];
}

// One axis of interpolate_fIn (LBMBlockComm.f90:808-914) at son index b
// (1-based; bT: the last odd index, bT + 1 the wrapped last column or row of
// an even count): the coarse indices and weights of
//   ((w0 F0 + w1 F1) + w2 F2) + w3 F3.
// Every pass of the reference is this sum: a copy (odd b), the one-sided sums
// at the ends, the central one (whose subtractions are additions of negated
// products), and for the linear scheme (F0 + F1) * 0.5 = 0.5 F0 + 0.5 F1.
// Weights that a sum leaves out are 0 on an index it uses.  One form for all
// nodes: as branches on the parities and ends, each with its own reads, a
// wave went through a dozen of them in turn.
template <int SCHEME>
struct Interp {
  static constexpr int N = SCHEME == 2 ? 4 : 2;
  int i[N];
  double w[N];
  __device__ __forceinline__ Interp(int b, int bT) {
    const int b1 = b / 2;  // the coarse index left of an even b
    if constexpr (SCHEME == 2) {
      const bool odd = b & 1, wrap = b > bT, lo = b == 2, hi = !lo && b == bT - 1;
      const bool side = !odd && !wrap && (lo || hi), mid = !odd && !side;
      const int d = hi ? -1 : 1;  // one-sided: from the nearest coarse index inward
      i[0] = odd ? (b + 1) / 2 : (wrap ? (bT - 1) / 2 : (side ? (hi ? b1 + 1 : b1) : b1 - 1));
      i[1] = odd ? i[0] : (wrap ? (bT + 1) / 2 : (side ? i[0] + d : b1));
      i[2] = odd ? i[0] : (wrap ? 1 : (side ? i[0] + 2 * d : b1 + 1));
      i[3] = odd || side ? i[0] : (wrap ? 2 : b1 + 2);
      w[0] = odd ? 1.0 : (mid ? -0.0625 : 0.375);
      w[1] = odd ? 0.0 : (mid ? 0.5625 : 0.75);
      w[2] = odd ? 0.0 : (mid ? 0.5625 : -0.125);
      w[3] = mid ? -0.0625 : 0.0;
    } else {
      const bool odd = b & 1, wrap = b > bT;
      i[0] = odd ? (b + 1) / 2 : (wrap ? (bT + 1) / 2 : b1);
      i[1] = odd ? i[0] : (wrap ? 1 : b1 + 1);
      w[0] = odd ? 1.0 : 0.5;
      w[1] = odd ? 0.0 : 0.5;
    }
  }
  __device__ __forceinline__ double sum(const double (&v)[N]) const {
    double s = w[0] * v[0];
#pragma unroll
    for (int k = 1; k < N; ++k) s = s + w[k] * v[k];
    return s;
  }
};

// Son plane node (b, a) (1-based) from the coarse plane p of one direction:
// along b first, then along a; the last column of an even b count is the sum
// along b of values already interpolated along a (LBMBlockComm.f90:862-868,
// 902-908), and its wrapped last row again along b first (:869-877, 909-913).
template <int SCHEME>
__device__ __forceinline__ double interp_node(const double *p, int bF, int b, int a, int aT, int bT) {
  using I = Interp<SCHEME>;
  const I ia(a, aT), ib(b, bT);
  double v[I::N][I::N], r[I::N];
#pragma unroll
  for (int j = 0; j < I::N; ++j)
#pragma unroll
    for (int k = 0; k < I::N; ++k) v[j][k] = p[(ia.i[j] - 1) * bF + (ib.i[k] - 1)];
  if (b > bT && a <= aT) {
#pragma unroll
    for (int k = 0; k < I::N; ++k) {
      double c[I::N];
#pragma unroll
      for (int j = 0; j < I::N; ++j) c[j] = v[j][k];
      r[k] = ia.sum(c);
    }
    return ib.sum(r);
  }
#pragma unroll
  for (int j = 0; j < I::N; ++j) r[j] = ib.sum(v[j]);
  return ia.sum(r);
}

// cell coordinates of in-plane (a, b) on a face of `axis` at `fixed`
__device__ __forceinline__ void plane_cell(int axis, int fixed, int a, int b, int &x, int &y, int &z) {
  if (axis == 0) { x = fixed; y = a; z = b; }
  else if (axis == 1) { x = a; y = fixed; z = b; }
  else { x = a; y = b; z = fixed; }
}

// extract_interpolate_layer (LBMBlockComm.f90:340-505): copy the father planes
// under the son's fluid faces; at level 2 also level1 = 0.5*(level1 + level2).
// grid: x over q*aF*bF of the largest face, y = face.
__global__ void k_tree_extract(TreeArgs t, int level) {
  const int face = blockIdx.y;
  const TreeFace &F = t.face[face];
  if (!F.active) return;
  const int np = F.aF * F.bF;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= Q * np) return;
  const int q = i / np, r = i - q * np;
  const int a = r / F.bF, b = r - a * F.bF;
  const int axis = face >> 1;
  const int oa = axis == 0 ? t.f0[1] : t.f0[0];
  const int ob = axis == 2 ? t.f0[1] : t.f0[2];
  int x, y, z;
  plane_cell(axis, F.fixedF, oa + a, ob + b, x, y, z);
  const double v = t.ff[(size_t)q * t.fN + ((size_t)x * t.fyd + y) * t.fzd + z];
  double *l1 = t.planes + F.off + i;
  if (level == 1) {
    *l1 = v;
  } else {
    l1[(size_t)Q * np] = v;
    *l1 = 0.5 * (*l1 + v);
  }
}

// is the son node (x, y, z) on an active son face after `face` in the
// reference's face order?  Later faces overwrite earlier ones there.
__device__ __forceinline__ bool later_face_owns(const TreeArgs &t, int face, int x, int y, int z, bool son) {
  bool owns = false;
#pragma unroll
  for (int g = 1; g < 6; ++g) {  // (all faces, so that their words are read together)
    const int c = (g >> 1) == 0 ? x : ((g >> 1) == 1 ? y : z);
    const int at = son ? t.face[g].fixedS : t.face[g].fixedFi;
    owns |= (g > face) & (t.face[g].active != 0) & (c == at);
  }
  return owns;
}

// interpolation_father_to_son (LBMBlockComm.f90:655-806): interpolate the
// coarse plane (level 1 at n_timeStep 0, level 2 at 1) onto the son boundary
// plane and rescale it with the father's volume force.
template <int SCHEME>
__global__ __launch_bounds__(kTreeNodes * Q) void k_tree_father_to_son(TreeArgs t, int level) {
  __shared__ double sh[Q][kTreeNodes];
  const int face = blockIdx.y;
  const TreeFace &F = t.face[face];
  if (!F.active || (int)blockIdx.x * kTreeNodes >= F.aS * F.bS) return;  // whole workgroups
  const int i = blockIdx.x * kTreeNodes + threadIdx.x, q = threadIdx.y;
  const int a0 = i / F.bS, b0 = i - a0 * F.bS;
  const int axis = face >> 1;
  int x, y, z;
  plane_cell(axis, F.fixedS, a0, b0, x, y, z);
  const bool on = i < F.aS * F.bS && !later_face_owns(t, face, x, y, z, true);
  if (on) {
    const int bT = (F.bS & 1) ? F.bS : F.bS - 1;
    const int aT = (F.aS & 1) ? F.aS : F.aS - 1;
    const size_t np = (size_t)F.aF * F.bF;
    const double *p = t.planes + F.off + (level == 2 ? (size_t)Q * np : 0) + q * np;
    sh[q][threadIdx.x] = interp_node<SCHEME>(p, F.bF, b0 + 1, a0 + 1, aT, bT);
  }
  __syncthreads();
  if (!on) return;
  double f[Q];
  tree_node(f, sh);
  t.fs[(size_t)q * t.sN + ((size_t)x * t.syd + y) * t.szd + z] = grid_transform(q, f, t.coeff, t.hv);
}

// deliver_son_to_father (LBMBlockComm.f90:546-653): every second son node of
// the son's first inner layer, rescaled with the son's volume force, replaces
// the father node it coincides with.
__global__ __launch_bounds__(kTreeNodes * Q) void k_tree_son_to_father(TreeArgs t) {
  __shared__ double sh[Q][kTreeNodes];
  const int face = blockIdx.y;
  const TreeFace &F = t.face[face];
  const int axis = face >> 1;
  const int ea = axis == 0 ? 1 : 0, eb = axis == 2 ? 1 : 2;  // in-plane axes
  const int na = t.sicnt[ea], nb = t.sicnt[eb];
  if (!F.active || (int)blockIdx.x * kTreeNodes >= na * nb) return;  // whole workgroups
  const int i = blockIdx.x * kTreeNodes + threadIdx.x, q = threadIdx.y;
  const int ia = i / nb, ib = i - ia * nb;
  int sx, sy, sz, fx, fy, fz;
  plane_cell(axis, F.fixedSi, t.si0[ea] + 2 * ia, t.si0[eb] + 2 * ib, sx, sy, sz);
  plane_cell(axis, F.fixedFi, t.fi0[ea] + ia, t.fi0[eb] + ib, fx, fy, fz);
  const bool on = i < na * nb && !later_face_owns(t, face, fx, fy, fz, false);
  if (on) sh[q][threadIdx.x] = t.fs[(size_t)q * t.sN + ((size_t)sx * t.syd + sy) * t.szd + sz];
  __syncthreads();
  if (!on) return;
  double f[Q];
  tree_node(f, sh);
  t.ff[(size_t)q * t.fN + ((size_t)fx * t.fyd + fy) * t.fzd + fz] = grid_transform(q, f, t.coeff, t.hv);
}

}  // namespace fsil
