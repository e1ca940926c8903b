// dk_stencil.hpp -- the point-particle stencil of the plain FP64 form (device functions shared by
// the per-particle kernels of dk_fp64.hip and the tile kernels of dk_tile64.hip).
#ifndef ATHENAK_AMD_CSRC_DK_STENCIL_HPP_
#define ATHENAK_AMD_CSRC_DK_STENCIL_HPP_

#include "dk_internal.hpp"

namespace dk {

struct Stencil {
  int ip, jp, kp;
  double wx[3], wy[3], wz[3];
};

__device__ inline void MakeStencil(const Geo &g, const DevBlock &b, double x, double y,
                                   double z, Stencil &w) {
  PMWeights(x, b.x1min, b.x1max, g.nx1, g.is, g.deposit, w.ip, w.wx);
  PMWeights(y, b.x2min, b.x2max, g.nx2, g.js, g.deposit, w.jp, w.wy);
  PMWeights(z, b.x3min, b.x3max, g.nx3, g.ks, g.deposit, w.kp, w.wz);
}

__device__ inline bool HaloOK(const Geo &g, const Stencil &w) {   // dust_pm.cpp:241-242
  return !(w.ip < (g.is-1) || w.ip > (g.is+g.nx1) || w.jp < (g.js-1) || w.jp > (g.js+g.nx2) ||
           w.kp < (g.ks-1) || w.kp > (g.ks+g.nx3));
}

// a stencil footprint must lie inside the padded block (guards every gather/deposit)
__device__ inline bool InPad(const Geo &g, const Stencil &w) {
  return w.ip >= 1 && w.ip <= g.n1 - 2 && w.jp >= 1 && w.jp <= g.n2 - 2 && w.kp >= 1 &&
         w.kp <= g.n3 - 2;
}

}  // namespace dk

#endif  // ATHENAK_AMD_CSRC_DK_STENCIL_HPP_
