// Device workspace of the implicit differentiation of window 0 (FP64), shared by its kernels and the host runtime.
#pragma once

#include <stdint.h>

namespace sba_dev {

constexpr int kAdjSlots = 256;  // workgroups of the passes over pairs, and slots of their partial sums

struct AdjData {
  int n6, nx, npf, pairs, obs;  // 6 ncf, 6 ncf + 3 npf, free points, pairs and observations of the window
  int tiles, slots;        // back-substitution tiles of the window, workgroups that share them
  int parity;              // conjugate-gradient iteration modulo 2
  double tol;
  double *spts, *sposes;                 // FP64 state: points [np][3], key frames [nc][12] (rows of [R | t])
  double *x, *r, *z, *p, *y, *gd;        // tangent vectors (nx)
  double *pc, *zc;                       // key-frame part of p (two buffers of 6 kMaxFreePoses), of S^-1 e
  double* jac;                           // per observation, value-major: J (2 x 9), the symmetric 2 x 2 weight (3)
  double *wh, *wg, *vh, *uh;             // blocks: 18 per pair, 18 per pair (value-major), 6 per point, 36 per key frame
  double *part, *part2;                  // key-frame partial sums per slot (27 ncf, 6 ncf)
  double *s_rz, *s_py, *s_rr, *sc;       // scalar slots; scalars (8)
  double *lst, *linv, *sinv;             // stored factor, its inverse, the inverse of the reduced system
  double *dxy, *dinfo;                   // per-observation gradients, the caller's order
  int32_t* done;
};

}  // namespace sba_dev
