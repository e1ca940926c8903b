// dk_tile64.hip -- tile kernels of the plain FP64 form: the particle-mesh passes of a stage
// (dust_pm.cpp:225-274, 500-564, 141-193, dust_solver.cpp:151-201, dust_push.cpp:132-245) over
// the caller's particle arrays, summed tile by tile in LDS.
//
// What bounds a per-particle deposit is its 81-108 FP64 atomic additions per particle: scattered
// over HBM they run at 25 G additions/s (a pass over 8.4 million particles took 25-33 ms), while
// the LDS adder takes a wavefront's 64 FP64 additions in 9 clocks (4.6 T/s over the chip) when
// its lanes hold different words.  So the particles are binned by tile (8 x 4 x 4 cells of a
// block): a histogram over the tiles with each particle's place in its tile, a scan, and a
// permutation; the arrays themselves stay in the caller's order.  A workgroup takes a tile's
// particles (an item: at most kItemMax of them) in chunks, groups a chunk by cell in LDS, gathers
// from an LDS copy of the tile and its halo, leaves one record per particle (its offsets in the
// cell and its values), and sums the records: a thread takes a run of at most kRun records of one
// cell and one x3 offset (slab) of the stencil, so that its 9 x NC sums stay in registers, and
// adds them into the tile's region in LDS.  The regions go to a scratch array that a combine pass
// adds up per cell; items after a tile's first, and the few particles whose centre cell lies
// outside the tile grid, add to the field directly.
//
// The order of a cell's additions is not fixed (as with the per-particle atomics).
//
// Fused multiply-adds only in the sums of the records (step 4, where they pay: without them the
// passes take 10 % longer): what a particle gathers and what becomes of it is rounded as on the
// per-particle kernels and in the reference's operation order, so that a particle's path does not
// depend on which kernels its deposit runs on (3 % of the gathering passes).
//
// Measured, per launch, per-particle kernels -> tile kernels with their combine: 8.4 million
// particles on 128^3 cells (shearing box), deposit of Q, P 33.5 -> 0.51 ms, operator 25.6 -> 0.58,
// kick 25.8 -> 0.69, the bins of a stage 0.12 ms; 2.1 million, half of them in clumps, 11.7 ->
// 0.15, 8.8 -> 0.16, 8.9 -> 0.18 ms; pc2 predictor and advance of 1 million in uneven blocks
// 5.5 -> 0.17 and 4.3 -> 0.15 ms.

#include <hip/hip_runtime.h>

#include <algorithm>

#include "dk_internal.hpp"
#include "dk_stencil.hpp"

using dk::DevBlock;
using dk::Geo;
using dk::Idx;
using dk::kBlock;
using dk::Stencil;

namespace {

constexpr int kTX = 8, kTY = 4, kTZ = 4, kTC = kTX*kTY*kTZ;   // cells of a tile
// threads of a tile kernel: one wavefront per SIMD, so that a CU holds as many workgroups as a SIMD
// holds wavefronts (three at the 130 to 167 registers of the nine sums of three or four values).
// Six wavefronts, one thread per (cell, slab), load two SIMDs twice: one workgroup a CU for the
// deposit and two for the others (8.4 million particles: deposit 0.83 -> 0.42, operator 0.63 ->
// 0.47, kick 0.84 -> 0.65 ms)
constexpr int kNT = 256;
// particles of a chunk: 512, the mean of a tile at 4 particles per cell, and three standard
// deviations of a random filling, so that such a tile is one chunk; with the records of 576 a
// workgroup takes 45 to 47 KB of LDS (50 to 53 KB in the shearing box), three on a CU.  (The pc2
// predictor, with a gathered field and four components, takes 55 and 62 KB: two.)
constexpr int kChunk = 576;
constexpr int kPer = (kChunk + kNT - 1)/kNT;
constexpr int kItemMax = 2*kChunk;
// records a thread sums before it adds to the region: longer runs add less often, shorter ones
// spread a crowded cell over more threads (2.1 million particles, half of them in clumps: the three
// passes 1.41 ms at 4, 1.08 at 6, 0.97 at 8, 0.86 at 12 and 16; even fillings alike from 6 on)
constexpr int kRun = 16;
// the centre cells of a tile's particles: its own, and in the shearing box those one row off in x2
// (every particle belongs to the tile of its cell clamped into the block)
constexpr int kCellMax = kTX*(kTY + 2)*kTZ;
constexpr int kRunMax = kCellMax + kChunk/kRun;

enum Op { kScatter = 0, kOper = 1, kKick = 2, kPredict = 3, kAdvance = 4 };

template <int OP> constexpr int NComp() { return (OP == kScatter || OP == kPredict) ? 4 : 3; }
template <int OP> constexpr bool Gathers() { return OP != kScatter; }

// the tiles of the mesh: ragged where a block's sides are no multiples of the tile's; the region
// of a tile adds a halo of one cell, in the shearing box one more in x2 on each side (a centre
// may sit one cell beyond a block's x2 face in the shifted frame)
struct Grid64 {
  int ntx, nty, ntz, ntb, nt, SY;
  int RX, RY, RZ, RN;
  float iRX, iRY;
};

struct Args64 {
  Geo g;
  Grid64 T;
  const DevBlock *B;
  double *r;
  const int32_t *iv;
  long long cap, np;
  const int *perm, *start, *item_tile, *item_part, *nitem;
  double sh, a_dt, dt;
  int rate_dep, sbox, strat;
  double qs, om;
  const double *src;      // u* (3 components), or u1 (the gas) for the predictor
  double *out;            // the field deposited into: nvar components, the first at comp0
  int nvar, comp0;
  double *scr;
  dk::ErrWord *err;
};

#define GRID_STRIDE(t, n) \
  for (long long t = blockIdx.x*(long long)blockDim.x + threadIdx.x; t < (n); \
       t += (long long)gridDim.x*blockDim.x)

inline int Grid(long long n) {
  long long b = (n + kBlock - 1)/kBlock;
  if (b < 1) b = 1;
  return static_cast<int>(std::min<long long>(b, 65536));
}

// i/d from the float reciprocal (0 <= i < 4096, d < 64, or i < 4 d)
__device__ inline int FDiv(int i, float inv) {
  return static_cast<int>((static_cast<float>(i) + 0.5f)*inv);
}

// PMWeights' centre cell (active index, unclamped) and offset along one axis
__device__ inline void Centre(double x, double lo, double sc, int &ic, double &del) {
#pragma clang fp contract(off)
  const double cell = (x - lo)*sc;
  ic = static_cast<int>(cell + 1.0) - 1;
  del = cell - (static_cast<double>(ic) + 0.5);
}

// where a particle deposits and gathers: its block, centre cell and offsets
struct Place {
  int m, ic, jc, kc;
  double dx, dy, dz;
};

// the position a pass works at: the particle's own with the frame shift sh x1 in x2
// (dust.hpp:1699-1702), or for the advance the half-step position (dust_push.cpp:150-155)
template <int OP>
__device__ inline Place Locate(const Args64 &A, long long p) {
#pragma clang fp contract(off)
  const double *r = A.r;
  const long long cap = A.cap;
  Place L;
  L.m = A.iv[(long long)DK_PGID*cap + p];
  const DevBlock &b = A.B[L.m];
  double x, y, z;
  if constexpr (OP == kAdvance) {
    const double x0 = r[(long long)DK_IPX1*cap + p], y0 = r[(long long)DK_IPY1*cap + p];
    const double z0 = r[(long long)DK_IPZ1*cap + p];
    x = x0 + 0.5*A.dt*r[(long long)DK_IPVX1*cap + p];
    const double yh = y0 + 0.5*A.dt*(r[(long long)DK_IPVY1*cap + p] -
                                     (A.sbox ? A.qs*A.om*x0 : 0.0));
    z = z0 + 0.5*A.dt*r[(long long)DK_IPVZ1*cap + p];
    y = yh + (A.sbox ? A.qs*A.om*x*0.5*A.dt : 0.0);
  } else {
    x = r[(long long)DK_IPX*cap + p];
    y = r[(long long)DK_IPY*cap + p] + A.sh*x;
    z = r[(long long)DK_IPZ*cap + p];
  }
  Centre(x, b.x1min, b.sx1, L.ic, L.dx);
  Centre(y, b.x2min, b.sx2, L.jc, L.dy);
  Centre(z, b.x3min, b.sx3, L.kc, L.dz);
  return L;
}

// the tile of a centre cell clamped into its block
__device__ inline int TileOf(const Geo &g, const Grid64 &T, const Place &L) {
  const int i = min(max(L.ic, 0), g.nx1 - 1), j = min(max(L.jc, 0), g.nx2 - 1);
  const int k = min(max(L.kc, 0), g.nx3 - 1);
  return ((L.m*T.ntz + k/kTZ)*T.nty + j/kTY)*T.ntx + i/kTX;
}

__device__ inline void Weights(int scheme, double d, double w[3]) {
#pragma clang fp contract(off)
  if (scheme == 2) {
    const double h0 = 0.5 - d, h2 = 0.5 + d;
    w[0] = 0.5*h0*h0; w[1] = 0.75 - d*d; w[2] = 0.5*h2*h2;
  } else if (scheme == 1) {
    w[0] = fmax(0.0, -d); w[1] = 1.0 - fabs(d); w[2] = fmax(0.0, d);
  } else {
    w[0] = 0.0; w[1] = 1.0; w[2] = 0.0;
  }
}

__device__ inline Stencil MakeW(const Geo &g, const Place &L) {
  Stencil w;
  w.ip = L.ic + g.is; w.jp = L.jc + g.js; w.kp = L.kc + g.ks;
  Weights(g.deposit, L.dx, w.wx);
  Weights(g.deposit, L.dy, w.wy);
  Weights(g.deposit, L.dz, w.wz);
  return w;
}

//----------------------------------------------------------------------------------------
// the bins

// every particle's tile and its place in the tile's count.  Particles sorted by cell put a
// wavefront's 64 particles into one to three tiles, in sparse blocks into more: one atomic per tile
// and wavefront, all of a wavefront's at once (one after another, each waiting for the last one's
// return, 1 million particles in uneven blocks took 50 us, now 39; 0.4 million in ragged blocks 18,
// now 10).
template <int OP>
__global__ void __launch_bounds__(kBlock) k_t64_count(Args64 A, int *key, int *rank, int *count) {
  const int lane = threadIdx.x & 63;
  const long long step = (long long)gridDim.x*kBlock;
  // (the loop bound is the wavefront's: every lane takes part in the ballots)
  for (long long p0 = (long long)blockIdx.x*kBlock + (threadIdx.x & ~63); p0 < A.np; p0 += step) {
    const long long p = p0 + lane;
    int t = -1;
    if (p < A.np) t = TileOf(A.g, A.T, Locate<OP>(A, p));
    unsigned long long pend = __ballot(t >= 0), mine = 0;
    int lead = lane;
    while (pend) {
      const int leader = __ffsll(static_cast<long long>(pend)) - 1;
      const int tl = __shfl(t, leader, 64);
      const unsigned long long peers = __ballot(t == tl);
      if (t == tl) {lead = leader; mine = peers;}
      pend &= ~peers;
    }
    int base = 0;
    if (t >= 0 && lane == lead) base = atomicAdd(&count[t], __popcll(mine));
    const int rk = __shfl(base, lead, 64) + __popcll(mine & ((1ull << lane) - 1ull));
    if (p < A.np) {key[p] = t; rank[p] = rk;}
  }
}

// inclusive prefix sum over a wavefront
__device__ inline int WaveScan(int v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int u = __shfl_up(v, d, 64);
    if (lane >= d) v += u;
  }
  return v;
}

// the tiles' first places and the items (at most kItemMax particles of one tile each, at least
// one per tile), in one workgroup: 4096 tiles per pass.  The counts are left cleared for the next
// bins.
constexpr int kScanThreads = 1024, kScanPer = 4;
__global__ void __launch_bounds__(kScanThreads)
k_t64_scan(int nt, int *count, int *start, int *item_tile, int *item_part, int *nitem) {
  __shared__ int wp[16], wi[16];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  int cp = 0, ci = 0;   // particles and items so far
  for (int t0 = 0; t0 < nt; t0 += kScanThreads*kScanPer) {
    int n[kScanPer], sp = 0, si = 0;
#pragma unroll
    for (int q=0; q<kScanPer; ++q) {
      const int t = t0 + tid*kScanPer + q;
      n[q] = 0;
      if (t < nt) {
        n[q] = count[t];
        count[t] = 0;
        si += max(1, (n[q] + kItemMax - 1)/kItemMax);
      }
      sp += n[q];
    }
    const int ap = WaveScan(sp), ai = WaveScan(si);
    if (lane == 63) {wp[wv] = ap; wi[wv] = ai;}
    __syncthreads();
    int bp = cp + ap - sp, bi = ci + ai - si;
    for (int w = 0; w < 16; ++w) {
      if (w < wv) {bp += wp[w]; bi += wi[w];}
      cp += wp[w]; ci += wi[w];
    }
#pragma unroll
    for (int q=0; q<kScanPer; ++q) {
      const int t = t0 + tid*kScanPer + q;
      if (t >= nt) break;
      start[t] = bp;
      bp += n[q];
      const int np = max(1, (n[q] + kItemMax - 1)/kItemMax);
      for (int k=0; k<np; ++k) {item_tile[bi + k] = t; item_part[bi + k] = k;}
      bi += np;
    }
    __syncthreads();   // (wp and wi are reused)
  }
  if (tid == 0) {start[nt] = cp; *nitem = ci;}
}

__global__ void k_t64_place(const int *key, const int *rank, const int *start, long long np,
                            int *perm) {
  GRID_STRIDE(p, np) perm[start[key[p]] + rank[p]] = static_cast<int>(p);
}

//----------------------------------------------------------------------------------------
// the tile kernels

// a particle whose centre cell lies outside the tile's cells, or whose numbers are not finite:
// gathered from and deposited into the padded fields directly (as the per-particle kernels)
template <int NC>
__device__ inline void FarDeposit(const Args64 &A, int m, const Stencil &w, const double val[NC]) {
  for (int c=0; c<3; ++c)
    for (int bb=0; bb<3; ++bb) {
      const double wcb = w.wz[c]*w.wy[bb];
      if (wcb == 0.0) continue;
      for (int a=0; a<3; ++a) {
        const double ww = wcb*w.wx[a];
        const long long i0 = Idx(A.g, m, A.nvar, A.comp0, w.kp+c-1, w.jp+bb-1, w.ip+a-1);
        for (int n=0; n<NC; ++n) unsafeAtomicAdd(&A.out[i0 + n*A.g.ncb], ww*val[n]);
      }
    }
}

template <int OP>
__device__ inline void FarGather(const Args64 &A, int m, const Stencil &w, double u[3]) {
#pragma clang fp contract(off)
  constexpr int nv = (OP == kPredict) ? DK_NGAS : 3;
  for (int d=0; d<3; ++d) u[d] = 0.0;
  for (int c=0; c<3; ++c)
    for (int bb=0; bb<3; ++bb) {
      const double wcb = w.wz[c]*w.wy[bb];
      if (wcb == 0.0) continue;
      for (int a=0; a<3; ++a) {
        double ww = wcb*w.wx[a];
        const long long i0 = Idx(A.g, m, nv, 0, w.kp+c-1, w.jp+bb-1, w.ip+a-1);
        if constexpr (OP == kPredict) {
          const double inv = 1.0/A.src[i0];
          for (int d=0; d<3; ++d) u[d] += ww*(A.src[i0 + (1 + d)*A.g.ncb]*inv);
        } else {
          for (int d=0; d<3; ++d) u[d] += ww*A.src[i0 + d*A.g.ncb];
        }
      }
    }
}

template <int N>
__device__ inline bool Finite(const double x[N]) {
  bool ok = true;
#pragma unroll
  for (int n=0; n<N; ++n) ok = ok && isfinite(x[n]);
  return ok;
}

// fac x; a particle without mass (fac 0) gives nothing whatever its velocity, as the per-particle
// kernels pass it over (the predictor's do not: its rate is no factor of the stencil's weights)
__device__ inline double Share(double fac, double x) { return (fac == 0.0) ? 0.0 : fac*x; }

// the particle's work of a pass: u, the gathered velocity; val, what it deposits per unit weight
template <int OP>
__device__ inline void Work(const Args64 &A, const DevBlock &b, long long p, const double u[3],
                            double *val) {
#pragma clang fp contract(off)
  double *r = A.r;
  const long long cap = A.cap;
  const double ts = r[(long long)DK_IPTS*cap + p], mass = r[(long long)DK_IPM*cap + p];
  const double vol = b.dx1*b.dx2*b.dx3;
  if constexpr (OP == kScatter) {
    const double muc = mass*(A.a_dt/(ts + A.a_dt))/vol;
    val[0] = muc;
    for (int d=0; d<3; ++d) val[1 + d] = Share(muc, r[(long long)(DK_IPVX + 2*d)*cap + p]);
  } else if constexpr (OP == kOper) {
    const double fac = mass*(A.a_dt/(ts + A.a_dt))/vol;
    for (int d=0; d<3; ++d) val[d] = Share(fac, u[d]);
  } else if constexpr (OP == kKick) {
    const double cj = A.a_dt/(ts + A.a_dt), fac = -mass/vol;
    for (int d=0; d<3; ++d) {
      double &v = r[(long long)(DK_IPVX + 2*d)*cap + p];
      const double dv = cj*(u[d] - v);
      v += dv;
      r[(long long)(DK_IPRX + d)*cap + p] = dv/A.a_dt;
      val[d] = Share(fac, dv);
    }
  } else if constexpr (OP == kPredict) {
    const double rate = mass/(ts*vol);
    for (int d=0; d<3; ++d)
      val[d] = -A.dt*rate*(u[d] - r[(long long)(DK_IPVX + 2*d)*cap + p]);
    val[3] = A.rate_dep ? rate : 0.0;
  } else {
    // the implicit-midpoint push (dust_push.cpp:160-230)
    const double dt = A.dt, h = 0.5*dt, lambda = h/ts, aa = 1.0 + lambda;
    double x0[3], v0[3], rr[3], vh[3], xh[3];
    for (int d=0; d<3; ++d) {
      x0[d] = r[(long long)(DK_IPX1 + 2*d)*cap + p];
      v0[d] = r[(long long)(DK_IPVX1 + 2*d)*cap + p];
      rr[d] = v0[d] + lambda*u[d];
    }
    xh[0] = x0[0] + 0.5*dt*v0[0];
    xh[1] = x0[1] + 0.5*dt*(v0[1] - (A.sbox ? A.qs*A.om*x0[0] : 0.0));
    xh[2] = x0[2] + 0.5*dt*v0[2];
    if (A.sbox) {
      const double cxy = 2.0*h*A.om, cyx = h*(2.0 - A.qs)*A.om, det = aa*aa + cxy*cyx;
      vh[0] = (aa*rr[0] + cxy*rr[1])/det;
      vh[1] = (aa*rr[1] - cyx*rr[0])/det;
      if (A.strat) rr[2] -= h*(A.om*A.om)*xh[2];
      vh[2] = rr[2]/aa;
    } else {
      for (int d=0; d<3; ++d) vh[d] = rr[d]/aa;
    }
    const double fac = -mass/vol;
    for (int d=0; d<3; ++d) {
      r[(long long)(DK_IPVX + 2*d)*cap + p] = 2.0*vh[d] - v0[d];
      const double drift = (d == 1 && A.sbox) ? vh[1] - A.qs*A.om*xh[0] : vh[d];
      r[(long long)(DK_IPX + 2*d)*cap + p] = x0[d] + dt*drift;
      r[(long long)(DK_IPX1 + 2*d)*cap + p] = xh[d];
      const double dv = dt*(u[d] - vh[d])/ts;
      r[(long long)(DK_IPRX + d)*cap + p] = dv;
      val[d] = Share(fac, dv);
    }
  }
}

// workgroups are handed to the 8 XCDs in turn: runs of kDeal consecutive items go to one XCD, so
// that neighbouring tiles (whose regions and fields overlap) share its L2, and the runs go round
// the XCDs, so that a crowded part of the mesh is spread over all of them
constexpr int kDeal = 32;
__device__ inline int Deal(int b, int n) {
  const int full = n/(8*kDeal)*(8*kDeal);
  if (b >= full) return b;
  const int x = b & 7, i = b >> 3;
  return ((i/kDeal)*8 + x)*kDeal + i % kDeal;
}

template <int OP>
__host__ __device__ constexpr size_t Lds64(int RN) {
  return sizeof(double)*((NComp<OP>() + (Gathers<OP>() ? 3 : 0))*(size_t)RN +
                         (3 + NComp<OP>())*(size_t)kChunk) +
         sizeof(int)*(2*kCellMax + kRunMax + 4);
}

template <int OP>
__global__ void __launch_bounds__(kNT, 3) k_t64(Args64 A) {
  constexpr int NC = NComp<OP>();
  extern __shared__ double lds[];
  const Geo &g = A.g;
  const Grid64 &T = A.T;
  const int it = Deal(blockIdx.x, gridDim.x);
  if (it >= *A.nitem) return;
  const int tile = A.item_tile[it], part = A.item_part[it];
  const int tid = threadIdx.x;
  const int m = tile/T.ntb;
  int q = tile - m*T.ntb;
  const int tx = q % T.ntx;
  q /= T.ntx;
  const int ty = q % T.nty, tz = q/T.nty;
  const int ci0 = tx*kTX, cj0 = ty*kTY, ck0 = tz*kTZ;
  const DevBlock &b = A.B[m];
  double *reg = lds;                                             // [NC][RN]
  double *us = reg + NC*T.RN;                                    // [3][RN]
  double *rec = us + (Gathers<OP>() ? 3*T.RN : 0);               // [3 + NC][kChunk]
  int *cnt = reinterpret_cast<int*>(rec + (3 + NC)*kChunk);      // [kCellMax]
  int *cst = cnt + kCellMax;                                     // [kCellMax]
  int *runs = cst + kCellMax;                                    // [kRunMax] cell | run << 8
  int *wt = runs + kRunMax;                                      // [4]
  const int NY = kTY + 2*T.SY, ncell = kTX*NY*kTZ;               // (a multiple of 64)
  for (int i = tid; i < NC*T.RN; i += kNT) reg[i] = 0.0;
  if (tid < ncell) cnt[tid] = 0;
  if constexpr (Gathers<OP>()) {
    for (int rc = tid; rc < T.RN; rc += kNT) {
      const int rr = FDiv(rc, T.iRX), rx = rc - rr*T.RX;
      const int rz = FDiv(rr, T.iRY), ry = rr - rz*T.RY;
      const int i = g.is + ci0 - 1 + rx, j = g.js + cj0 - 1 - T.SY + ry, k = g.ks + ck0 - 1 + rz;
      double v[3] = {0.0, 0.0, 0.0};
      if (i < g.n1 && j < g.n2 && k < g.n3) {   // (a ragged tile's region passes the block's end)
        if constexpr (OP == kPredict) {
          const long long i0 = Idx(g, m, DK_NGAS, DK_IDN, k, j, i);
          const double inv = 1.0/A.src[i0];
          for (int d=0; d<3; ++d) v[d] = A.src[i0 + (1 + d)*g.ncb]*inv;
        } else {
          const long long i0 = Idx(g, m, 3, 0, k, j, i);
          for (int d=0; d<3; ++d) v[d] = A.src[i0 + d*g.ncb];
        }
      }
      for (int d=0; d<3; ++d) us[d*T.RN + rc] = v[d];
    }
  }
  const int s0 = A.start[tile] + part*kItemMax, s1 = min(A.start[tile + 1], s0 + kItemMax);
  const int nch = (s1 - s0 + kChunk - 1)/kChunk;
  const int per = (nch > 0) ? (s1 - s0 + nch - 1)/nch : 1;
  __syncthreads();
  for (int c0 = s0; c0 < s1; c0 += per) {
    const int n = min(per, s1 - c0);
    // 1. every particle's cell in the tile and its place among the chunk's particles there
    Place L[kPer];
    int p[kPer], cell[kPer], rk[kPer];
#pragma unroll
    for (int k=0; k<kPer; ++k) {
      const int i = tid + k*kNT;
      cell[k] = -1;
      p[k] = -1;
      if (i < n) {
        p[k] = A.perm[c0 + i];
        L[k] = Locate<OP>(A, p[k]);
        const int li = L[k].ic - ci0, lk = L[k].kc - ck0;
        const int lj = L[k].jc - cj0 + T.SY;
        const bool near = li >= 0 && li < kTX && L[k].ic < g.nx1 && lk >= 0 && lk < kTZ &&
                          L[k].kc < g.nx3 && lj >= 0 && lj < NY && L[k].jc >= -T.SY &&
                          L[k].jc < g.nx2 + T.SY;
        if (near) {
          cell[k] = (lk*NY + lj)*kTX + li;
          rk[k] = atomicAdd(&cnt[cell[k]], 1);
        }
      }
    }
    __syncthreads();
    // 2. the cells' first places and the runs
    int nc = 0, ap = 0;
    if (tid < ncell) {
      nc = cnt[tid];
      ap = WaveScan(nc | (((nc + kRun - 1)/kRun) << 16));
      if ((tid & 63) == 63) wt[tid >> 6] = ap;
    }
    __syncthreads();
    const int nruns = (wt[0] >> 16) + (wt[1] >> 16) + (T.SY ? (wt[2] >> 16) : 0);
    if (tid < ncell) {
      if (tid >= 64) ap += wt[0];
      if (tid >= 128) ap += wt[1];
      const int nr = (nc + kRun - 1)/kRun;
      cst[tid] = (ap & 0xffff) - nc;
      for (int k=0; k<nr; ++k) runs[(ap >> 16) - nr + k] = tid | (k << 8);
    }
    __syncthreads();
    // 3. the particles' work and their records
#pragma unroll
    for (int k=0; k<kPer; ++k) {
      if (p[k] < 0) continue;
      double val[NC];
      double u[3] = {0.0, 0.0, 0.0};
      const bool far = cell[k] < 0;
      if (__builtin_expect(far, 0)) {
        // outside the tile's cells: inside the padded block only
        const Stencil w = MakeW(g, L[k]);
        if (!((OP == kScatter) ? dk::HaloOK(g, w) : dk::InPad(g, w))) {
          dk::RecordError(A.err, DK_EHALO, p[k]);
          continue;
        }
      }
      if constexpr (Gathers<OP>()) {
        if (!far) {
#pragma clang fp contract(off)
          double wx[3], wy[3], wz[3];
          Weights(g.deposit, L[k].dx, wx);
          Weights(g.deposit, L[k].dy, wy);
          Weights(g.deposit, L[k].dz, wz);
          const int rb = ((L[k].kc - ck0)*T.RY + (L[k].jc - cj0 + T.SY))*T.RX + (L[k].ic - ci0);
#pragma unroll
          for (int c=0; c<3; ++c)
#pragma unroll
            for (int bb=0; bb<3; ++bb) {
              const double wcb = wz[c]*wy[bb];
              const int row = rb + (c*T.RY + bb)*T.RX;
#pragma unroll
              for (int a=0; a<3; ++a) {
                const double ww = wcb*wx[a];
#pragma unroll
                for (int d=0; d<3; ++d) u[d] += ww*us[d*T.RN + row + a];
              }
            }
        }
        // The sums over the tile multiply the rows of weight zero too, which the per-particle
        // kernels pass over: the same for finite numbers.  So a particle that gathers or gives
        // what is not finite goes their way.
        if (__builtin_expect(far || !Finite<3>(u), 0)) FarGather<OP>(A, m, MakeW(g, L[k]), u);
      }
      Work<OP>(A, b, p[k], u, val);
      const bool direct = far || !Finite<NC>(val);
      if (__builtin_expect(direct, 0)) FarDeposit<NC>(A, m, MakeW(g, L[k]), val);
      if (far) continue;
      const int at = cst[cell[k]] + rk[k];
      rec[at] = L[k].dx; rec[kChunk + at] = L[k].dy; rec[2*kChunk + at] = L[k].dz;
#pragma unroll
      for (int v=0; v<NC; ++v) rec[(3 + v)*kChunk + at] = direct ? 0.0 : val[v];
    }
    __syncthreads();
    // 4. the runs' sums, per slab, into the region
    for (int task = tid; task < 3*nruns; task += kNT) {
      const int slab = (task >= 2*nruns) ? 2 : ((task >= nruns) ? 1 : 0);
      const int rn = runs[task - slab*nruns];
      const int l = rn & 255, a0 = cst[l] + (rn >> 8)*kRun;
      const int a1 = min(a0 + kRun, cst[l] + cnt[l]);
      double acc[3][3][NC];
#pragma unroll
      for (int bb=0; bb<3; ++bb)
#pragma unroll
        for (int a=0; a<3; ++a)
#pragma unroll
          for (int v=0; v<NC; ++v) acc[bb][a][v] = 0.0;
      for (int at = a0; at < a1; ++at) {
        double wx[3], wy[3], wz[3];
        Weights(g.deposit, rec[at], wx);
        Weights(g.deposit, rec[kChunk + at], wy);
        Weights(g.deposit, rec[2*kChunk + at], wz);
        const double ws = (slab == 0) ? wz[0] : ((slab == 1) ? wz[1] : wz[2]);
        double val[NC];
#pragma unroll
        for (int v=0; v<NC; ++v) val[v] = rec[(3 + v)*kChunk + at];
#pragma unroll
        for (int bb=0; bb<3; ++bb) {
          const double wcb = ws*wy[bb];
#pragma unroll
          for (int a=0; a<3; ++a) {
            const double ww = wcb*wx[a];
#pragma unroll
            for (int v=0; v<NC; ++v) acc[bb][a][v] += ww*val[v];
          }
        }
      }
      const int lx = l & (kTX - 1), lr = l/kTX, lz = lr/NY, ly = lr - lz*NY;
      const int rb = ((lz + slab)*T.RY + ly)*T.RX + lx;
#pragma unroll
      for (int bb=0; bb<3; ++bb)
#pragma unroll
        for (int a=0; a<3; ++a)
#pragma unroll
          for (int v=0; v<NC; ++v)
            unsafeAtomicAdd(&reg[v*T.RN + rb + bb*T.RX + a], acc[bb][a][v]);
    }
    __syncthreads();
    if (tid < ncell) cnt[tid] = 0;
    __syncthreads();
  }
  // the region: the tile's first item to the scratch, row by row (the rows of the tiles of a block
  // that share ty and tz lie one after another), a later one straight into the field
  for (int rc = tid; rc < T.RN; rc += kNT) {
    const int rr = FDiv(rc, T.iRX), rx = rc - rr*T.RX;
    const int rz = FDiv(rr, T.iRY), ry = rr - rz*T.RY;
    if (part == 0) {
      const long long row = (((((long long)m*T.ntz + tz)*T.nty + ty)*NC)*T.RZ + rz)*T.RY + ry;
      const long long at = row*T.ntx*T.RX + tx*T.RX + rx;
      const long long vs = (long long)T.RZ*T.RY*T.ntx*T.RX;
#pragma unroll
      for (int v=0; v<NC; ++v) A.scr[at + v*vs] = reg[v*T.RN + rc];
    } else {
      const int i = g.is + ci0 - 1 + rx, j = g.js + cj0 - 1 - T.SY + ry, k = g.ks + ck0 - 1 + rz;
      if (i < g.n1 && j < g.n2 && k < g.n3) {
        const long long i0 = Idx(g, m, A.nvar, A.comp0, k, j, i);
#pragma unroll
        for (int v=0; v<NC; ++v) {
          const double s = reg[v*T.RN + rc];
          if (s != 0.0) unsafeAtomicAdd(&A.out[i0 + v*g.ncb], s);
        }
      }
    }
  }
}

// every padded cell adds the first items' regions of the tiles that cover it to what the later
// items and the particles outside their tile have left in the field (x: a block's cells, y: blocks)
template <int NC>
__global__ void __launch_bounds__(kBlock) k_t64_combine(Geo g, Grid64 T, const double *scr,
                                                        double *out, int nvar, int comp0) {
  const int m = blockIdx.y;
  const unsigned ncb = static_cast<unsigned>(g.ncb);
  for (unsigned rr = blockIdx.x*blockDim.x + threadIdx.x; rr < ncb; rr += gridDim.x*blockDim.x) {
    const unsigned t2 = rr/static_cast<unsigned>(g.n1);
    const unsigned k_ = t2/static_cast<unsigned>(g.n2);
    const int i = static_cast<int>(rr - t2*g.n1), j = static_cast<int>(t2 - k_*g.n2);
    const int k = static_cast<int>(k_);
    // the cell in the coordinates of tile 0's region
    const int ai = i - g.is + 1, aj = j - g.js + 1 + T.SY, ak = k - g.ks + 1;
    if (ai < 0 || aj < 0 || ak < 0) continue;
    const int tz0 = max(0, (ak - T.RZ + kTZ)/kTZ), tz1 = min(T.ntz - 1, ak/kTZ);
    const int ty0 = max(0, (aj - T.RY + kTY)/kTY), ty1 = min(T.nty - 1, aj/kTY);
    const int tx0 = max(0, (ai - T.RX + kTX)/kTX), tx1 = min(T.ntx - 1, ai/kTX);
    double sum[NC];
#pragma unroll
    for (int v=0; v<NC; ++v) sum[v] = 0.0;
    const long long vs = (long long)T.RZ*T.RY*T.ntx*T.RX;
    for (int tz=tz0; tz<=tz1; ++tz) {
      const int rz = ak - tz*kTZ;
      if (rz >= T.RZ) continue;
      for (int ty=ty0; ty<=ty1; ++ty) {
        const int ry = aj - ty*kTY;
        if (ry >= T.RY) continue;
        for (int tx=tx0; tx<=tx1; ++tx) {
          const int rx = ai - tx*kTX;
          if (rx >= T.RX) continue;
          const long long row = (((((long long)m*T.ntz + tz)*T.nty + ty)*NC)*T.RZ + rz)*T.RY + ry;
          const long long at = row*T.ntx*T.RX + tx*T.RX + rx;
#pragma unroll
          for (int v=0; v<NC; ++v) sum[v] += scr[at + v*vs];
        }
      }
    }
#pragma unroll
    for (int v=0; v<NC; ++v) out[Idx(g, m, nvar, comp0 + v, k, j, i)] += sum[v];
  }
}

}  // namespace

// the workspaces of the present particles: the items and every particle's tile, place and slot
struct Bins64 {
  int *item_tile = nullptr, *item_part = nullptr, *key = nullptr, *rank = nullptr, *perm = nullptr;
  void *mem = nullptr;      // the one allocation that holds them (null: Tile64's, the first ones)
  long long cap = 0;        // particles they hold
  // A graph that the caller captured holds them: they stay until the context ends, also when more
  // particles are bound, so that the graph may be replayed as before (its particles and the
  // context's fields outlive a bind as well).  prev: the ones kept so.
  bool captured = false;
  Bins64 *prev = nullptr;
};

// the workspaces of a context's tile passes; those of the mesh are allocated once, the first
// particles' with them
struct Tile64 {
  Grid64 T;
  int *count = nullptr, *start = nullptr, *nitem = nullptr;
  double *scr = nullptr;
  void *mem = nullptr;      // the one allocation that holds them
  Bins64 *b = nullptr;
  int bins = 0;             // the bins of the present positions are built (T64Hold)
};

namespace dk {

namespace {

// the caller is capturing the context's stream (the library's own stage graphs, which are captured
// anew before every launch, apart)
bool CallerCaptures(const dk_ctx *c) {
  if (c->own_capture) return false;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(c->stream, &cs) == hipSuccess) return cs != hipStreamCaptureStatusNone;
  (void)hipGetLastError();
  return true;
}

// While another stream is captured, in any mode but the relaxed one, this thread's allocations and
// waits would be refused and end that capture; they are no part of it.
struct Relaxed {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  Relaxed() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  ~Relaxed() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

// one allocation (null: short of device memory, and then the per-particle kernels run)
void *Mem(size_t bytes) {
  void *p = nullptr;
  if (hipMalloc(&p, bytes) == hipSuccess) return p;
  (void)hipGetLastError();
  return nullptr;
}

Args64 MakeArgs(const dk_ctx *c, double sh, double a_dt, double dt) {
  const Tile64 *w = c->t64;
  Args64 A{};
  A.g = c->g; A.T = w->T; A.B = c->d_blocks;
  A.r = c->rdata; A.iv = c->idata; A.cap = c->cap; A.np = c->np;
  A.perm = w->b->perm; A.start = w->start; A.nitem = w->nitem;
  A.item_tile = w->b->item_tile; A.item_part = w->b->item_part;
  A.sh = sh; A.a_dt = a_dt; A.dt = dt;
  A.sbox = c->P.shearing_box; A.strat = c->P.stratified;
  A.qs = c->P.qshear; A.om = c->P.omega0;
  A.scr = w->scr; A.err = c->d_err;
  return A;
}

template <int OP>
int Bin(dk_ctx *c, const Args64 &A) {
  Tile64 *w = c->t64;
  Bins64 *b = w->b;
  if (c->stream != nullptr && CallerCaptures(c)) b->captured = true;
  const int pt = ProfBegin(c, "bins");
  k_t64_count<OP><<<Grid(c->np), kBlock, 0, c->stream>>>(A, b->key, b->rank, w->count);
  k_t64_scan<<<1, kScanThreads, 0, c->stream>>>(w->T.nt, w->count, w->start, b->item_tile,
                                                b->item_part, w->nitem);
  k_t64_place<<<Grid(c->np), kBlock, 0, c->stream>>>(b->key, b->rank, w->start, c->np, b->perm);
  ProfEnd(c, pt);
  return Check(hipGetLastError());
}

// one pass: the bins (unless the caller holds them), the tile kernel, the combine into out's
// NC components from comp0
template <int OP>
int Pass(dk_ctx *c, Args64 A, const char *label) {
  Tile64 *w = c->t64;
  int e;
  if (!w->bins && (e = Bin<OP>(c, A))) return e;
  constexpr int NC = NComp<OP>();
  const long long items = (long long)w->T.nt + c->np/kItemMax;
  {const int pt = ProfBegin(c, label);
   k_t64<OP><<<static_cast<unsigned>(items), kNT, Lds64<OP>(w->T.RN), c->stream>>>(A);
   ProfEnd(c, pt);}
  {const int pt = ProfBegin(c, "combine");
   const dim3 gr(static_cast<unsigned>((c->g.ncb + kBlock - 1)/kBlock), c->g.nmb);
   k_t64_combine<NC><<<gr, kBlock, 0, c->stream>>>(c->g, w->T, A.scr, A.out, A.nvar, A.comp0);
   ProfEnd(c, pt);}
  return Check(hipGetLastError());
}

Grid64 MakeGrid(const dk_ctx *c) {
  Grid64 T;
  const Geo &g = c->g;
  T.SY = c->P.shearing_box ? 1 : 0;
  T.ntx = (g.nx1 + kTX - 1)/kTX; T.nty = (g.nx2 + kTY - 1)/kTY; T.ntz = (g.nx3 + kTZ - 1)/kTZ;
  T.ntb = T.ntx*T.nty*T.ntz;
  T.nt = static_cast<int>(std::min<long long>((long long)T.ntb*g.nmb, INT32_MAX));
  T.RX = kTX + 2; T.RY = kTY + 2 + 2*T.SY; T.RZ = kTZ + 2;
  T.RN = T.RX*T.RY*T.RZ;
  T.iRX = 1.0f/T.RX; T.iRY = 1.0f/T.RY;
  return T;
}

// The tile passes cost every tile's region and the combine whatever the particles, the
// per-particle kernels their atomics.  A step (imex2+ / pc2), tile passes against per-particle
// kernels: 128^3 cells at 8 particles a tile (one per 16 cells) 3.08 against 4.14 / 1.51 against 1.73
// ms, at 4 a tile 2.97 against 2.47 / 1.47 against 1.01.  Where blocks leave tiles partly empty it
// is the particles a tile that count: 4096 blocks of 4^3 cells at 4 a tile 1.07 against 1.05 / 0.46
// against 0.41 ms, at 8 1.07 against 1.35 / 0.46 against 0.50; 343 blocks of 9^3 at 5 a tile 0.89
// against 1.08 / 0.39 against 0.38; 2197 blocks of 5^3 at 4 1.41 against 1.39 / 0.62 against 0.50,
// at 8 1.44 against 2.04 / 0.63 against 0.69; 32768 blocks of 2^3 at 2 6.95 against 5.41 / 2.94
// against 2.18, at 8 7.19 against 9.11 / 2.99 against 3.31.
// Without back-reaction nothing is deposited, and the per-particle kernels gather alone: sorted
// particles, kick or advance of a step on the tile passes (their bins, and sums that nobody reads)
// against the per-particle kernel, 33 thousand 47 against 19 us, 2.1 million in clumps 0.35 against
// 0.23 ms, 67 million 8.9 against 8.1, pc2 7.5 million in uneven blocks 0.78 against 0.61.  (In no order
// within their blocks the tile passes' gather was the faster one for large even boxes, 67 million 43
// against 83 ms, and the slower one for small boxes, clumps and uneven blocks.)
bool Pays(const dk_ctx *c, const Grid64 &T) {
  if (!c->P.back_reaction) return false;
  const long long a_tile = (c->P.coupling == DK_PC2) ? 6 : 5;
  return c->np*16 >= (long long)c->g.nmb*c->g.nx1*c->g.nx2*c->g.nx3 && c->np >= a_tile*T.nt;
}

// the particles' part of the workspaces, for n of them: its ints, and its place at p
size_t BinsInts(const Grid64 &T, long long n) {
  return 2*static_cast<size_t>(T.nt + n/kItemMax + 1) + 3*static_cast<size_t>(n);
}

Bins64 *MakeBins(const Grid64 &T, long long n, int *p) {
  const size_t items = static_cast<size_t>(T.nt + n/kItemMax + 1);
  Bins64 *b = new Bins64();
  b->item_tile = p;
  b->item_part = b->item_tile + items;
  b->key = b->item_part + items;
  b->rank = b->key + n;
  b->perm = b->rank + n;
  b->cap = n;
  return b;
}

// the mesh's part with the first particles', for n of them, in one allocation (two take 0.3 ms more
// of a small program's start); false: short of device memory
bool First(dk_ctx *c, const Grid64 &T, long long n) {
  const long long nt = T.nt;
  // the scratch, then the int arrays
  const size_t nscr = 4*(size_t)T.RN*nt, nmesh = 2*(size_t)(nt + 1) + 1;
  void *mem = Mem(sizeof(double)*nscr + sizeof(int)*(nmesh + BinsInts(T, n)));
  if (mem == nullptr) return false;
  Tile64 *w = new Tile64();
  w->T = T;
  w->mem = mem;
  w->scr = static_cast<double*>(mem);
  w->count = reinterpret_cast<int*>(w->scr + nscr);
  w->start = w->count + nt + 1;
  w->nitem = w->start + nt + 1;
  w->b = MakeBins(T, n, w->nitem + 1);
  c->t64 = w;
  return true;
}

}  // namespace

int T64Reserve(dk_ctx *c) {
  if (c->form != DK_FORM_FP64 || c->smr || c->P.clouds || c->g.ng < 2) return DK_OK;
  const Grid64 T = MakeGrid(c);
  if (!Pays(c, T) || T.nt >= (1 << 29)) return DK_OK;   // (32-bit items)
  if (c->t64 != nullptr && c->t64->b->cap >= c->np) return DK_OK;
  if (CallerCaptures(c))
    return DK_OK;   // (no allocation inside the caller's capture: the per-particle kernels run)
  const Relaxed relaxed;
  // for as many as the caller's arrays hold, so that a count that grows within them neither
  // allocates nor waits (12 of their 156 bytes a particle)
  long long n = std::min<long long>(c->cap, INT32_MAX);
  if (c->t64 == nullptr) {
    if (!First(c, T, n) && !First(c, T, c->np)) return DK_OK;
    const int e = Check(hipMemsetAsync(c->t64->count, 0, sizeof(int)*(T.nt + 1), c->stream));
    if (e) T64Destroy(c);
    return e;
  }
  Tile64 *w = c->t64;
  Bins64 *old = w->b;
  if (old->captured) {
    // (half as many again as the ones kept, so that what growing arrays leave behind stays below
    // twice what they have)
    n = std::max(n, std::min<long long>(old->cap + old->cap/2, INT32_MAX));
  } else if (old->mem != nullptr) {
    (void)hipStreamSynchronize(c->stream);
    w->b = old->prev;
    (void)hipFree(old->mem);
    delete old;
  }
  void *mem = Mem(sizeof(int)*BinsInts(T, n));
  if (mem == nullptr && n > c->np) mem = Mem(sizeof(int)*BinsInts(T, n = c->np));
  if (mem == nullptr) return DK_OK;
  Bins64 *b = MakeBins(T, n, static_cast<int*>(mem));
  b->mem = mem;
  b->prev = w->b;
  w->b = b;
  return DK_OK;
}

void T64Destroy(dk_ctx *c) {
  Tile64 *w = c->t64;
  if (w == nullptr) return;
  while (w->b != nullptr) {
    Bins64 *b = w->b;
    w->b = b->prev;
    if (b->mem != nullptr) (void)hipFree(b->mem);
    delete b;
  }
  (void)hipFree(w->mem);
  delete w;
  c->t64 = nullptr;
}

bool T64Yield(dk_ctx *c) {
  if (c->t64 == nullptr || c->t64->bins || CallerCaptures(c)) return false;
  for (const Bins64 *b = c->t64->b; b != nullptr; b = b->prev)
    if (b->captured) return false;
  (void)hipStreamSynchronize(c->stream);
  T64Destroy(c);
  return true;
}

bool T64Use(const dk_ctx *c) {
  return c->t64 != nullptr && c->t64->b->cap >= c->np && Pays(c, c->t64->T);
}

int T64Hold(dk_ctx *c, double sh) {
  if (!T64Use(c)) return DK_OK;
  const int e = Bin<kScatter>(c, MakeArgs(c, sh, 0.0, 0.0));
  if (!e) c->t64->bins = 1;
  return e;
}

bool T64Held(const dk_ctx *c) { return c->t64 != nullptr && c->t64->bins != 0; }

void T64Release(dk_ctx *c) {
  if (c->t64 != nullptr) c->t64->bins = 0;
}

int T64Scatter(dk_ctx *c, double a_dt, double sh) {
  Args64 A = MakeArgs(c, sh, a_dt, 0.0);
  A.out = c->qdep; A.nvar = 5; A.comp0 = 0;
  return Pass<kScatter>(c, A, "scatter_imex");
}

int T64Oper(dk_ctx *c, const double *field, double *out, double a_dt, double sh) {
  Args64 A = MakeArgs(c, sh, a_dt, 0.0);
  A.src = field; A.out = out; A.nvar = 3; A.comp0 = 0;
  return Pass<kOper>(c, A, "applya_gtsg");
}

int T64Kick(dk_ctx *c, double a_dt, double sh) {
  Args64 A = MakeArgs(c, sh, a_dt, 0.0);
  A.src = c->ustar; A.out = c->dmom; A.nvar = 3; A.comp0 = 0;
  return Pass<kKick>(c, A, "gather_kick");
}

int T64Predictor(dk_ctx *c, double dt, int rate_dep) {
  Args64 A = MakeArgs(c, 0.0, 0.0, dt);
  A.src = c->u1; A.out = c->qdep; A.nvar = 5; A.comp0 = 1;
  A.rate_dep = rate_dep;
  return Pass<kPredict>(c, A, "pc2_predictor");
}

int T64Advance(dk_ctx *c, double dt) {
  Args64 A = MakeArgs(c, 0.0, 0.0, dt);
  A.src = c->ustar; A.out = c->dmom; A.nvar = 3; A.comp0 = 0;
  return Pass<kAdvance>(c, A, "pc2_advance");
}

}  // namespace dk
