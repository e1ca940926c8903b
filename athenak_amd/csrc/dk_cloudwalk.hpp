// dk_cloudwalk.hpp -- the refinable cloud's shape and its walk over the leaves of a statically
// refined mesh (device code shared by the FP64 form's cloud kernels and the FP32 form's
// cross-level clouds).
#ifndef ATHENAK_AMD_CSRC_DK_CLOUDWALK_HPP_
#define ATHENAK_AMD_CSRC_DK_CLOUDWALK_HPP_

#include <cmath>

#include "dk_internal.hpp"
#include "dk_smr.hpp"

namespace dk {

// the cloud half-width (the root cell size) per direction, its reciprocal, the mesh lengths
struct CloudGeo {
  double h[3], ih[3], len[3];
};

__device__ inline double Sq(double x) { return x*x; }

// src/dust/dust.hpp:169-182 (CloudGeometry::HatCDF, HatMoment)
__device__ inline double HatCDF(const double s) {
  if (s <= -1.0) return 0.0;
  if (s >= 1.0) return 1.0;
  return (s <= 0.0) ? 0.5*Sq(1.0 + s) : 1.0 - 0.5*Sq(1.0 - s);
}
__device__ inline double HatMoment(const double s) {
  if (s <= -1.0 || s >= 1.0) return 1.0/6.0;
  return (s <= 0.0) ? 0.5*Sq(s) + Sq(s)*s/3.0 : 0.5*Sq(s) - Sq(s)*s/3.0;
}
// src/dust/dust.hpp:186-188
__device__ inline double MinImage(const double d, const double length) {
  return d - length*round(d/length);
}

// LeafTraversal3D::ForEach (src/dust/dust_leaf3d.hpp:383-517) on a statically refined mesh: the
// actual leaves under the cloud of level lev at x (half-width root dx 2^-lev) at their own
// resolution, by a group of kCoop lanes of one wavefront per cloud.  The candidates are the leaves
// holding the support's 8 corners (a leaf at least as long as the support in every direction
// meets it only if it holds a corner); the walk is refused when a corner lies in no leaf or a
// candidate is shorter than the support.
//
// One thread per cloud is a chain of dependent loads (eight corner searches, then each leaf cell's
// pack) at one to three wavefronts per SIMD, its atomics scattered over as many clouds as lanes.
// Here eight lanes find the corners' leaves at once, the cells of all leaves are numbered in one
// sequence and the lanes take them in turn, so that a cloud's loads are in flight together and
// neighbouring lanes touch neighbouring cells.  A cell's weight and moments come from its own two
// faces per axis.  (792 blocks of 16^3, 9.7 million clouds at 3 per cell, FP64: predictor 56 -> 31 ms,
// advance 45 -> 25 ms; 13 million in the FP32 form: its cross-level clouds 11 -> 6.3 ms a step.)
constexpr int kCoop = 32;
struct CoopLeaf {
  double b0[3], d[3];   // the leaf's lower corner in the cloud's frame, its cell sizes
  int b, start;         // the leaf, the number of its first cell in the sequence
  int c0[3], n[3];      // its first cell under the cloud and the cells per axis
};
struct CoopCloud {
  double h[3], ih[3];
  int total;            // cells of all leaves; negative: the walk is refused
};

// lane: the thread's place in its group; lf: the group's 8 entries in LDS.  Every lane of the
// group calls it.
__device__ inline CoopCloud CoopSpans(const Geo &g, const DevBlock *B, const SmrTree &t,
                                      const CloudGeo &cg, const double x[3], const int lev,
                                      const int lane, CoopLeaf *lf) {
  CoopCloud cl;
  double lo[3], hi[3], p[3];
  int k[3];
  const int c = lane & 7;
#pragma unroll
  for (int d=0; d<3; ++d) {
    cl.h[d] = ldexp(cg.h[d], -lev);
    cl.ih[d] = ldexp(cg.ih[d], lev);
    lo[d] = x[d] - cl.h[d];
    hi[d] = x[d] + cl.h[d];
    p[d] = ((c >> d) & 1) ? nextafter(hi[d], -INFINITY) : lo[d];
  }
  SmrWrap(t, p, k);
  const int b = SmrLeafAt(B, t, p);
  bool bad = b < 0, dup = false;
#pragma unroll
  for (int q=0; q<7; ++q) {
    const int ob = __shfl(b, q, 8), o0 = __shfl(k[0], q, 8), o1 = __shfl(k[1], q, 8);
    const int o2 = __shfl(k[2], q, 8);
    if (q < c && ob == b && o0 == k[0] && o1 == k[1] && o2 == k[2]) dup = true;
  }
  CoopLeaf me{};
  me.b = b;
  int n = 0;
  if (!bad) {
    const DevBlock &bb = B[b];
    const double bl[3] = {bb.x1min, bb.x2min, bb.x3min}, bh[3] = {bb.x1max, bb.x2max, bb.x3max};
    const double dd[3] = {bb.dx1, bb.dx2, bb.dx3};
    const int nx[3] = {g.nx1, g.nx2, g.nx3};
    n = dup ? 0 : 1;
#pragma unroll
    for (int d=0; d<3; ++d) {
      if (bh[d] - bl[d] < 2.0*cl.h[d]) bad = true;
      me.d[d] = dd[d];
      me.b0[d] = bl[d] + k[d]*cg.len[d];
      const double id = 1.0/dd[d];
      const int i0 = max(static_cast<int>(floor((lo[d] - me.b0[d])*id)), 0);
      const int i1 = min(static_cast<int>(ceil((hi[d] - me.b0[d])*id)) - 1, nx[d] - 1);
      me.c0[d] = i0;
      me.n[d] = max(i1 - i0 + 1, 0);
      n *= me.n[d];
    }
  }
  int s = n;
#pragma unroll
  for (int d = 1; d < 8; d <<= 1) {
    const int u = __shfl_up(s, d, 8);
    if (c >= d) s += u;
  }
  me.start = s - n;
  cl.total = __shfl(s, 7, 8);
  const unsigned long long group = ((1ull << kCoop) - 1ull) << ((threadIdx.x & 63) & ~(kCoop - 1));
  if (__ballot(bad) & group) cl.total = -1;
  __builtin_amdgcn_wave_barrier();
  if (lane < 8) lf[c] = me;
  // (one wavefront: its LDS operations complete in order; the fence holds the compiler to it)
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  return cl;
}

// the lane's cells: f(leaf entry, k, j, i, w, m1x, m1y, m1z) with moments (unpadded indices),
// f(leaf entry, k, j, i, w) without
template <bool kMoments, class F>
__device__ inline void CoopCells(const CoopCloud &cl, const CoopLeaf *lf, const double x[3],
                                 const int lane, const F &f) {
  for (int c = lane; c < cl.total; c += kCoop) {
    int q = 0;
#pragma unroll
    for (int u=1; u<8; ++u)
      if (lf[u].start <= c) q = u;
    const CoopLeaf &L = lf[q];
    const int r = c - L.start, row = r/L.n[0];
    int id[3];
    id[0] = r - row*L.n[0];
    id[2] = row/L.n[1];
    id[1] = row - id[2]*L.n[1];
    double w[3], m[3];
#pragma unroll
    for (int d=0; d<3; ++d) {
      id[d] += L.c0[d];
      const double sa = (L.b0[d] + id[d]*L.d[d] - x[d])*cl.ih[d];
      const double sb = (L.b0[d] + (id[d] + 1)*L.d[d] - x[d])*cl.ih[d];
      w[d] = HatCDF(sb) - HatCDF(sa);
      if (kMoments) m[d] = cl.h[d]*(HatMoment(sb) - HatMoment(sa));
    }
    const double w23 = w[1]*w[2], wt = w23*w[0];
    if constexpr (kMoments) {
      const double m1x = w23*m[0], m1y = w[0]*m[1]*w[2], m1z = w[0]*w[1]*m[2];
      if (wt == 0.0 && m1x == 0.0 && m1y == 0.0 && m1z == 0.0) continue;
      f(L, id[2], id[1], id[0], wt, m1x, m1y, m1z);
    } else {
      if (wt == 0.0) continue;
      f(L, id[2], id[1], id[0], wt);
    }
  }
}

// A group takes a run of consecutive clouds, which in sorted order are mostly clouds of one cell: a
// lane keeps the sums of its leaf cell in registers while the next cloud gives it the same one, and
// adds them when it changes.  (The walk is bound by its atomic additions: one per cloud, cell and
// value took 10.7 of the FP32 form's 18.4 ms in three steps of a refined mesh with uneven blocks;
// now 11.6 in all.  FP64 form, 792 blocks of 16^3: predictor 31.6 -> 12.9, advance 24.4 -> 17.0 ms.)
// The run: 16, or less where there are too few clouds to give 16384 groups one.
__device__ inline int CoopRun(long long n) {
  return static_cast<int>(min(16LL, max(1LL, n >> 14)));
}

template <int NV, typename TO>
struct CoopHeld {
  long long at = -1;   // the word held, -1: none
  double v[NV];
  // (the values first to last - 1 are in use, ncb words apart)
  __device__ void Flush(TO *out, long long ncb, int first, int last) {
    if (at < 0) return;
    for (int d=first; d<last; ++d) unsafeAtomicAdd(&out[at + d*ncb], static_cast<TO>(v[d]));
  }
  // the sums of word i0: those of another word are added first
  __device__ void Take(TO *out, long long ncb, int first, int last, long long i0) {
    if (at == i0) return;
    Flush(out, ncb, first, last);
    at = i0;
    for (int d=0; d<NV; ++d) v[d] = 0.0;
  }
};

// the coefficients of the linear gather (LeafApi<LeafTraversal3D>::GatherLinear,
// src/dust/dust_leaf_api.hpp:202-220) in a cell: (first moment + (x - x_cell) w)/(2 dx) per axis
__device__ inline void CoopLinear(const CoopLeaf &L, const int k, const int j, const int i,
                                  const double w, const double m1x, const double m1y,
                                  const double m1z, const double x[3], double cf[3]) {
  cf[0] = 0.5*(m1x + (x[0] - (L.b0[0] + (i + 0.5)*L.d[0]))*w)/L.d[0];
  cf[1] = 0.5*(m1y + (x[1] - (L.b0[1] + (j + 0.5)*L.d[1]))*w)/L.d[1];
  cf[2] = 0.5*(m1z + (x[2] - (L.b0[2] + (k + 0.5)*L.d[2]))*w)/L.d[2];
}

// the sum over the group's lanes, in every lane
__device__ inline double CoopSum(double v) {
#pragma unroll
  for (int o = kCoop/2; o > 0; o >>= 1) v += __shfl_xor(v, o, kCoop);
  return v;
}

inline CloudGeo MakeCloudGeo(const dk_ctx *c) {
  CloudGeo cg;
  const dk_mesh &M = c->M;
  // the root cell size (src/dust/dust_cloud.cpp:135, dust_cloud3d.cpp:591-593)
  cg.h[0] = (M.x1max - M.x1min)/static_cast<double>(M.nmbx1*M.nx1);
  cg.h[1] = (M.x2max - M.x2min)/static_cast<double>(M.nmbx2*M.nx2);
  cg.h[2] = (M.x3max - M.x3min)/static_cast<double>(M.nmbx3*M.nx3);
  for (int d=0; d<3; ++d) cg.ih[d] = 1.0/cg.h[d];
  cg.len[0] = M.x1max - M.x1min;
  cg.len[1] = M.x2max - M.x2min;
  cg.len[2] = M.x3max - M.x3min;
  return cg;
}

}  // namespace dk

#endif  // ATHENAK_AMD_CSRC_DK_CLOUDWALK_HPP_
