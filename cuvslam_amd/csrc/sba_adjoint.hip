// Implicit gradient through a converged SBA solve (FP64), on the device.
//
// At a solution x* of min_x F(x; theta), F = sum_o rho(r_o^T L_o r_o), r_o = xy_o - pi(x), the gradient
// g(x*, theta) = grad_x F vanishes. For a loss of the solution, dL/dtheta = -a^T dg/dtheta with H a = dL/dx,
// H the full Hessian of F at x* (rho'' terms and the second-order terms of the projection and of the
// left-multiplied twist included). Tangent coordinates: left twists (omega, v) of the free key frames, then
// the free points, as the solver's own step. The observation parameters are xy_o and the symmetric L_o; a
// caller maps them to pixels and intrinsics (x = (u - c_x)/f_x, L_xy = diag(f) L_uv diag(f),
// libs/camera/observation.cpp:57-67).
//
// H a = g is solved by preconditioned conjugate gradients. The preconditioner is the Gauss-Newton system
// 2 sum rho' J^T L J of the converged state, solved through its Schur complement with the reduced camera
// system factored once in FP64 (the solver's own k_schur / k_reduce / k_factor at lambda = 0).
// An observation couples one key frame and one point, so H and the Gauss-Newton system are block-sparse: 6 x 6 blocks
// per key frame, 3 x 3 per point and one 6 x 3 block W per (point, key frame) pair. k_adj_assemble forms, once per state,
// these blocks for the preconditioner and for the second-order part of H, and for the first-order part of H each
// observation's J and 2 x 2 weight: J v is formed per observation, because along the weakly determined directions (the
// scale of a window) the key frames' and the points' parts of J v cancel, and summing their products with assembled
// blocks first would lose those digits (the gradients then differed by 1e-9 instead of 1e-12). A product is a pass over
// these numbers instead of a new FP64 linearization of every observation. A conjugate-gradient iteration is four
// launches: k_adj_hvp (y = H p), k_adj_update (x, r, and the Schur right-hand side), k_adj_reduced (the key-frame part,
// dense) and k_adj_precond (z). Each workgroup owns whole points and adds over key frames into its own slot (atomically
// in shared memory, so the last bits of two runs can differ); the scalars of an iteration are sums of one slot per
// workgroup, taken in the same order by every workgroup that needs them. 180k
// observations, 18 free key frames, microseconds per launch: 15.6 + 10.9 + 13.9 + 8.8 an iteration, 31.5 to assemble;
// with a linearization of every observation per product (FP64 atomics on the points) and the vector algebra in
// one workgroup, an iteration was seven launches of 47 + 15.5 + 12.6 + 15 + 42 + 15.5 + 15.5. The passes are bound by the
// loads of their 312 (Hessian) and 144 bytes per pair. No reference counterpart (the reference has no differentiation);
// its analytic Jacobians (schur_complement_bundler_cpu.cpp:101-118) are the anchors.
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>

#include "sba_adjoint.h"
#include "sba_device.h"
#include "sba_tiles.h"

using namespace sba_dev;

namespace {

constexpr double kHither64 = static_cast<double>(0.1f);  // epipolar/near_plane.h:33-38

__device__ __forceinline__ double drho64(int kind, double s, double d) {
  if (kind == 0) return (d + 1.0) / (d + s);
  if (d <= 0.0 || s < d * d) return 0.5;
  return 0.5 * d / sqrt(s);
}

__device__ __forceinline__ double d2rho64(int kind, double s, double d) {
  if (kind == 0) return -(d + 1.0) / ((d + s) * (d + s));
  if (d <= 0.0 || s < d * d) return 0.0;
  return -0.25 * d / (s * sqrt(s));
}

struct Lin64 {
  double r[2], J[2][9], L[3], w, w2, q0[3], P[3], Rcr[3][3], Rrw[3][3], D1[3][9];
};

// FP64 linearization of one observation at the FP64 state: p_r = T_rw p, p_c = T_cr p_r, J = dproj D1 with
// D1 = R_cr [-[p_r]x, I, R_rw] (the tangent of a left twist of T_rw and of the point).
__device__ bool lin64(const double* pose, const float4* cam, const double* X, float2 xy, float4 inf, int kind,
                      double delta, Lin64& o) {
  const float4 cr[3] = {cam[0], cam[1], cam[2]};
  for (int a = 0; a < 3; ++a) {
    const double* row = pose + 4 * a;
    const double crow[4] = {cr[a].x, cr[a].y, cr[a].z, cr[a].w};
    for (int k = 0; k < 3; ++k) {
      o.Rrw[a][k] = row[k];
      o.Rcr[a][k] = crow[k];
    }
    o.q0[a] = row[0] * X[0] + row[1] * X[1] + row[2] * X[2] + row[3];
  }
  const double tc[3] = {cr[0].w, cr[1].w, cr[2].w};
  for (int a = 0; a < 3; ++a) o.P[a] = o.Rcr[a][0] * o.q0[0] + o.Rcr[a][1] * o.q0[1] + o.Rcr[a][2] * o.q0[2] + tc[a];
  if (!(o.P[2] > kHither64)) return false;
  const double iz = 1.0 / o.P[2], u = o.P[0] * iz, v = o.P[1] * iz;
  o.r[0] = static_cast<double>(xy.x) - u;
  o.r[1] = static_cast<double>(xy.y) - v;
  const double mq[3][3] = {{0, o.q0[2], -o.q0[1]}, {-o.q0[2], 0, o.q0[0]}, {o.q0[1], -o.q0[0], 0}};
  for (int a = 0; a < 3; ++a)
    for (int k = 0; k < 3; ++k) {
      double s1 = 0, s3 = 0;
      for (int m = 0; m < 3; ++m) {
        s1 += o.Rcr[a][m] * mq[m][k];
        s3 += o.Rcr[a][m] * o.Rrw[m][k];
      }
      o.D1[a][k] = s1;
      o.D1[a][3 + k] = o.Rcr[a][k];
      o.D1[a][6 + k] = s3;
    }
  for (int k = 0; k < 9; ++k) {
    o.J[0][k] = iz * (o.D1[0][k] - u * o.D1[2][k]);
    o.J[1][k] = iz * (o.D1[1][k] - v * o.D1[2][k]);
  }
  o.L[0] = inf.x;
  o.L[1] = inf.y;
  o.L[2] = inf.z;
  const double Lr0 = o.L[0] * o.r[0] + o.L[1] * o.r[1], Lr1 = o.L[1] * o.r[0] + o.L[2] * o.r[1];
  const double s = o.r[0] * Lr0 + o.r[1] * Lr1;
  o.w = drho64(kind, s, delta);
  o.w2 = d2rho64(kind, s, delta);
  return true;
}

__device__ __forceinline__ void cross3(const double a[3], const double b[3], double o[3]) {
  o[0] = a[1] * b[2] - a[2] * b[1];
  o[1] = a[2] * b[0] - a[0] * b[2];
  o[2] = a[0] * b[1] - a[1] * b[0];
}

// The second-order part of h = H_o v for one observation (9 tangent entries: pose twist, point); the rest of H_o is
// J^T (2 rho' L + 4 rho'' L r r^T L) J.
__device__ __forceinline__ void hess2_obs(const Lin64& L, const double v[9], double h[9]) {
  const double Lr[2] = {L.L[0] * L.r[0] + L.L[1] * L.r[1], L.L[1] * L.r[0] + L.L[2] * L.r[1]};
  // - 2 Hess(c^T pi) v, c = rho' L r: D1^T Hpi D1 v plus the second-order terms of p_r along v
  const double c[2] = {L.w * Lr[0], L.w * Lr[1]};
  const double iz = 1.0 / L.P[2];
  const double g3[3] = {c[0] * iz, c[1] * iz, -(c[0] * L.P[0] + c[1] * L.P[1]) * iz * iz};
  double dv[3] = {0, 0, 0};
  for (int a = 0; a < 3; ++a)
    for (int k = 0; k < 9; ++k) dv[a] += L.D1[a][k] * v[k];
  const double hd[3] = {-c[0] * iz * iz * dv[2], -c[1] * iz * iz * dv[2],
                        -c[0] * iz * iz * dv[0] - c[1] * iz * iz * dv[1] +
                            2 * (c[0] * L.P[0] + c[1] * L.P[1]) * iz * iz * iz * dv[2]};
  double hpsi[9];
  for (int k = 0; k < 9; ++k) hpsi[k] = L.D1[0][k] * hd[0] + L.D1[1][k] * hd[1] + L.D1[2][k] * hd[2];
  double gp[3];
  for (int m = 0; m < 3; ++m) gp[m] = L.Rcr[0][m] * g3[0] + L.Rcr[1][m] * g3[1] + L.Rcr[2][m] * g3[2];
  double Rdp[3];
  for (int m = 0; m < 3; ++m) Rdp[m] = L.Rrw[m][0] * v[6] + L.Rrw[m][1] * v[7] + L.Rrw[m][2] * v[8];
  double wxq[3], avec[3], gxw[3], t1[3], t2[3];
  cross3(v, L.q0, wxq);
  for (int m = 0; m < 3; ++m) avec[m] = 0.5 * wxq[m] + 0.5 * v[3 + m] + Rdp[m];
  cross3(avec, gp, t1);
  cross3(gp, v, gxw);
  cross3(L.q0, gxw, t2);
  for (int m = 0; m < 3; ++m) {
    hpsi[m] += t1[m] + 0.5 * t2[m];
    hpsi[3 + m] += 0.5 * gxw[m];
    hpsi[6 + m] += L.Rrw[0][m] * gxw[0] + L.Rrw[1][m] * gxw[1] + L.Rrw[2][m] * gxw[2];
  }
  for (int k = 0; k < 9; ++k) h[k] = -2 * hpsi[k];
}

// Sum over the workgroup's 256 threads in every thread, in a fixed order; sh holds 4 doubles. Two barriers.
__device__ __forceinline__ double block_sum(double x, double* sh) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
  __syncthreads();  // sh is free
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = x;
  __syncthreads();
  return (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// Sum of one slot per workgroup, in every thread.
__device__ __forceinline__ double slot_sum(const double* slots, int n, double* sh) {
  double x = 0.0;
  for (int k = threadIdx.x; k < n; k += kBlock) x += slots[k];
  return block_sum(x, sh);
}

// V*^-1 q of point i (written by the Schur kernel at lambda = 0).
__device__ __forceinline__ void apply_vinv(const Batch& b, int i, const double q[3], double out[3]) {
  const float4 a0 = b.paux[3 * i], a1 = b.paux[3 * i + 1];
  const double Vi[3][3] = {{a0.x, a0.y, a0.z}, {a0.y, a0.w, a1.x}, {a0.z, a1.x, a1.y}};
  for (int a = 0; a < 3; ++a) out[a] = Vi[a][0] * q[0] + Vi[a][1] * q[1] + Vi[a][2] * q[2];
}

// This thread's pair of a back-substitution tile of window 0.
struct PairOf {
  int pair, point, key_frame;  // point inside the tile
  bool valid, coupled;         // coupled: a free point seen from a free key frame (it has a W block)
};
__device__ __forceinline__ PairOf pair_of(const Batch& b, const Tile& T, int npf, int ncf) {
  PairOf p{T.pair_begin + static_cast<int>(threadIdx.x), 0, 0, false, false};
  p.valid = p.pair < T.pair_end;
  if (p.valid) {
    const int z = b.pair_rec[p.pair].z;
    p.point = z >> 16;
    p.key_frame = z & 0xffff;
    p.coupled = T.point_begin + p.point < npf && p.key_frame < ncf;
  }
  return p;
}

}  // namespace

// The state-dependent numbers of window 0 at its FP64 state, and the gradient of its cost: per pair W of the
// Gauss-Newton system (w J_c^T L J_p, half the preconditioner) and, with HESS, per observation J and the weight
// 2 rho' L + 4 rho'' L r r^T L, and the second-order part of the Hessian as W per pair, V per point and U per key frame
// (hess2_obs of unit vectors). One thread per pair; point sums in pair order through shared memory, key-frame sums
// (21 of U, 6 of the gradient) per workgroup, added over the workgroups by k_adj_gather. FP64 arithmetic bounds it.
template <bool HESS>
__global__ __launch_bounds__(kBlock) void k_adj_assemble(Batch b, AdjData A) {
  __shared__ double sPoint[9 * kBlock];  // per pair: its part of V (6) and of the gradient (3)
  __shared__ double sPose[27 * kMaxFreePoses];
  const WindowDesc W = b.win[0];
  const int tid = threadIdx.x, ncf = W.ncf, npf = W.npf;
  const double delta = W.robust;
  for (int k = tid; k < 27 * ncf; k += kBlock) sPose[k] = 0.0;
  const int t0 = (A.tiles * blockIdx.x) / A.slots, t1 = (A.tiles * (blockIdx.x + 1)) / A.slots;
  for (int t = t0; t < t1; ++t) {
    const Tile T = b.btiles[t];
    const PairOf q = pair_of(b, T, npf, ncf);
    __syncthreads();  // sPose cleared; the previous tile's sPoint is free
    if (q.valid) {
      const int i = T.point_begin + q.point, j = q.key_frame;
      const bool pf = i < npf, cf = j < ncf;
      double V[6] = {}, gp[3] = {}, wh[18] = {}, wg[18] = {};
      const int4 rec = b.pair_rec[q.pair];
      for (int o = rec.x; o < rec.y; ++o) {
        const float4 inf = b.obs_info[o];
        Lin64 L;
        if (!lin64(A.sposes + 12 * j, b.cams + 3 * __float_as_int(inf.w), A.spts + 3 * i, b.obs_xy[o], inf, b.loss, delta,
                   L)) {
          if (HESS)
            for (int k = 0; k < 21; ++k) A.jac[static_cast<int64_t>(k) * A.obs + o] = 0.0;
          continue;
        }
        // grad F = -2 sum rho' J^T L r
        const double Lr[2] = {L.L[0] * L.r[0] + L.L[1] * L.r[1], L.L[1] * L.r[0] + L.L[2] * L.r[1]};
        if (cf)
          for (int k = 0; k < 6; ++k)
            atomicAdd(&sPose[27 * j + 21 + k], -2 * L.w * (L.J[0][k] * Lr[0] + L.J[1][k] * Lr[1]));
        if (pf) {
          for (int k = 0; k < 3; ++k) gp[k] -= 2 * L.w * (L.J[0][6 + k] * Lr[0] + L.J[1][6 + k] * Lr[1]);
          if (cf)
            for (int k = 0; k < 3; ++k) {
              const double l0 = L.w * (L.L[0] * L.J[0][6 + k] + L.L[1] * L.J[1][6 + k]);
              const double l1 = L.w * (L.L[1] * L.J[0][6 + k] + L.L[2] * L.J[1][6 + k]);
              for (int r = 0; r < 6; ++r) wg[3 * r + k] += L.J[0][r] * l0 + L.J[1][r] * l1;
            }
        }
        if (HESS) {
          const double m[3] = {2 * L.w * L.L[0] + 4 * L.w2 * Lr[0] * Lr[0], 2 * L.w * L.L[1] + 4 * L.w2 * Lr[0] * Lr[1],
                               2 * L.w * L.L[2] + 4 * L.w2 * Lr[1] * Lr[1]};
#pragma unroll
          for (int k = 0; k < 9; ++k) {
            A.jac[static_cast<int64_t>(k) * A.obs + o] = L.J[0][k];
            A.jac[static_cast<int64_t>(9 + k) * A.obs + o] = L.J[1][k];
          }
          for (int k = 0; k < 3; ++k) A.jac[static_cast<int64_t>(18 + k) * A.obs + o] = m[k];
          double e[9] = {}, h[9];
          if (cf) {
            int u = 0;
#pragma unroll
            for (int k = 0; k < 6; ++k) {
              e[k] = 1.0;
              hess2_obs(L, e, h);
              e[k] = 0.0;
#pragma unroll
              for (int r = 0; r <= k; ++r) atomicAdd(&sPose[27 * j + u++], h[r]);
            }
          }
          if (pf) {
            int u = 0;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
              e[6 + k] = 1.0;
              hess2_obs(L, e, h);
              e[6 + k] = 0.0;
#pragma unroll
              for (int r = 0; r < 6; ++r) wh[3 * r + k] += h[r];
#pragma unroll
              for (int r = 0; r <= k; ++r) V[u++] += h[6 + r];
            }
          }
        }
      }
      for (int k = 0; k < 6; ++k) sPoint[k * kBlock + tid] = V[k];
      for (int k = 0; k < 3; ++k) sPoint[(6 + k) * kBlock + tid] = gp[k];
      if (q.coupled)
        for (int k = 0; k < 18; ++k) {
          A.wg[static_cast<int64_t>(k) * A.pairs + q.pair] = wg[k];
          if (HESS) A.wh[static_cast<int64_t>(k) * A.pairs + q.pair] = wh[k];
        }
    }
    __syncthreads();
    const int i = T.point_begin + tid;
    if (i < T.point_end && i < npf) {
      const int qa = b.point_pair[i] - T.pair_begin, qe = min(b.point_pair[i + 1] - T.pair_begin, kBlock);
      double s[9] = {};
      for (int q2 = qa; q2 < qe; ++q2)
        for (int k = 0; k < 9; ++k) s[k] += sPoint[k * kBlock + q2];
      if (HESS)
        for (int k = 0; k < 6; ++k) A.vh[static_cast<int64_t>(k) * npf + i] = s[k];
      for (int k = 0; k < 3; ++k) A.gd[A.n6 + 3 * i + k] = s[6 + k];
    }
  }
  __syncthreads();
  for (int k = tid; k < 27 * ncf; k += kBlock) A.part[static_cast<int64_t>(blockIdx.x) * 27 * ncf + k] = sPose[k];
}

// Key-frame sums of k_adj_assemble: U (6 x 6, both triangles) and the gradient. One workgroup per value.
__global__ __launch_bounds__(kBlock) void k_adj_gather(Batch b, AdjData A, int hess) {
  __shared__ double sh[4];
  const int ncf = b.win[0].ncf, e = blockIdx.x, j = e / 27, v = e % 27;
  double x = 0.0;
  for (int g = threadIdx.x; g < A.slots; g += kBlock) x += A.part[static_cast<int64_t>(g) * 27 * ncf + e];
  x = block_sum(x, sh);
  if (threadIdx.x != 0) return;
  if (v >= 21) {
    A.gd[6 * j + v - 21] = x;
  } else if (hess) {
    int c = 0, r = v;  // column c of the upper triangle, rows 0..c
    while (r > c) r -= ++c;
    A.uh[36 * j + 6 * r + c] = x;
    A.uh[36 * j + 6 * c + r] = x;
  }
}

// Per-observation gradients of the converged solution from its adjoint v (tangent), in the caller's observation order.
__global__ __launch_bounds__(kBlock) void k_adj_obs_grad(Batch b, AdjData A, const int32_t* obs_orig) {
  const WindowDesc W = b.win[0];
  const int ncf = W.ncf, npf = W.npf;
  const double delta = W.robust;
  const Tile T = b.btiles[blockIdx.x];
  const PairOf q = pair_of(b, T, npf, ncf);
  if (!q.valid) return;
  const int i = T.point_begin + q.point, j = q.key_frame;
  const int4 rec = b.pair_rec[q.pair];
  for (int o = rec.x; o < rec.y; ++o) {
    const float4 inf = b.obs_info[o];
    Lin64 L;
    const bool valid = lin64(A.sposes + 12 * j, b.cams + 3 * __float_as_int(inf.w), A.spts + 3 * i, b.obs_xy[o], inf,
                             b.loss, delta, L);
    const int oo = obs_orig[o];
    double* gx = A.dxy + 2 * oo;
    double* gi = A.dinfo + 3 * oo;
    gx[0] = gx[1] = gi[0] = gi[1] = gi[2] = 0.0;
    if (!valid) continue;
    double av[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    if (j < ncf)
      for (int k = 0; k < 6; ++k) av[k] = A.x[6 * j + k];
    if (i < npf)
      for (int k = 0; k < 3; ++k) av[6 + k] = A.x[A.n6 + 3 * i + k];
    double Ja[2] = {0, 0};
    for (int k = 0; k < 9; ++k) {
      Ja[0] += L.J[0][k] * av[k];
      Ja[1] += L.J[1][k] * av[k];
    }
    const double LJa[2] = {L.L[0] * Ja[0] + L.L[1] * Ja[1], L.L[1] * Ja[0] + L.L[2] * Ja[1]};
    const double Lr[2] = {L.L[0] * L.r[0] + L.L[1] * L.r[1], L.L[1] * L.r[0] + L.L[2] * L.r[1]};
    const double rLJa = L.r[0] * LJa[0] + L.r[1] * LJa[1];
    gx[0] = 2 * (L.w * LJa[0] + 2 * L.w2 * rLJa * Lr[0]);
    gx[1] = 2 * (L.w * LJa[1] + 2 * L.w2 * rLJa * Lr[1]);
    const double G00 = 2 * (L.w * Ja[0] * L.r[0] + L.w2 * rLJa * L.r[0] * L.r[0]);
    const double G01 = 2 * (L.w * Ja[0] * L.r[1] + L.w2 * rLJa * L.r[0] * L.r[1]);
    const double G10 = 2 * (L.w * Ja[1] * L.r[0] + L.w2 * rLJa * L.r[1] * L.r[0]);
    const double G11 = 2 * (L.w * Ja[1] * L.r[1] + L.w2 * rLJa * L.r[1] * L.r[1]);
    gi[0] = G00;
    gi[1] = G01 + G10;
    gi[2] = G11;
  }
}

// ---- conjugate gradients: iteration `it` (from 0) of H x = gd ------------------------------------------------------
// Scalars: sc[0] |g|^2, sc[1] |r|^2, sc[2] iterations done, sc[4 + it % 2] r.z before iteration it. Slots: s_rz, s_py,
// s_rr, one per workgroup.

// p = z + beta p, y = H p, and the workgroups' shares of p.y and of the key-frame part of y. Every workgroup forms
// the key-frame part of p itself; it is kept in two buffers, so that none overwrites what another still reads.
__global__ __launch_bounds__(kBlock) void k_adj_hvp(Batch b, AdjData A, int it) {
  __shared__ double sPc[6 * kMaxFreePoses], sPose[6 * kMaxFreePoses];
  __shared__ double sP[3 * kBlock], sPair[3 * kBlock];
  __shared__ double sh[4];
  if (*A.done) return;
  const WindowDesc W = b.win[0];
  const int tid = threadIdx.x, ncf = W.ncf, npf = W.npf, n6 = A.n6;
  const double rz = A.sc[3] + slot_sum(A.s_rz, A.slots, sh);
  const double beta = it == 0 ? 0.0 : rz / A.sc[4 + ((it + 1) & 1)];
  if (blockIdx.x == 0 && tid == 0) A.sc[4 + (it & 1)] = rz;
  const double* pc_old = A.pc + 6 * kMaxFreePoses * ((it + 1) & 1);
  double* pc_new = A.pc + 6 * kMaxFreePoses * (it & 1);
  for (int k = tid; k < n6; k += kBlock) {
    const double v = it == 0 ? A.z[k] : A.z[k] + beta * pc_old[k];
    sPc[k] = v;
    sPose[k] = 0.0;
    if (blockIdx.x == 0) pc_new[k] = v;
  }
  double py = 0.0;
  const int t0 = (A.tiles * blockIdx.x) / A.slots, t1 = (A.tiles * (blockIdx.x + 1)) / A.slots;
  for (int t = t0; t < t1; ++t) {
    const Tile T = b.btiles[t];
    const PairOf q = pair_of(b, T, npf, ncf);
    double w[18], jac[21];
    int4 rec = make_int4(0, 0, 0, 0);
    if (q.valid) {
      rec = b.pair_rec[q.pair];
#pragma unroll
      for (int k = 0; k < 21; ++k) jac[k] = A.jac[static_cast<int64_t>(k) * A.obs + rec.x];
    }
    if (q.coupled) {
#pragma unroll
      for (int k = 0; k < 18; ++k) w[k] = A.wh[static_cast<int64_t>(k) * A.pairs + q.pair];
    }
    const int i = T.point_begin + tid;
    const bool point = i < T.point_end && i < npf;
    double p[3] = {};
    if (point) {
      const int at = n6 + 3 * i;
      for (int k = 0; k < 3; ++k) {
        p[k] = it == 0 ? A.z[at + k] : A.z[at + k] + beta * A.p[at + k];
        A.p[at + k] = p[k];
        sP[3 * tid + k] = p[k];
      }
    }
    __syncthreads();
    if (q.valid) {
      const bool cf = q.key_frame < ncf, pf = T.point_begin + q.point < npf;
      double c[6], pp[3], s[3] = {}, e[6] = {};
#pragma unroll
      for (int r = 0; r < 6; ++r) c[r] = cf ? sPc[6 * q.key_frame + r] : 0.0;
#pragma unroll
      for (int k = 0; k < 3; ++k) pp[k] = pf ? sP[3 * q.point + k] : 0.0;
      if (q.coupled) {
#pragma unroll
        for (int r = 0; r < 6; ++r) {
#pragma unroll
          for (int k = 0; k < 3; ++k) s[k] += w[3 * r + k] * c[r];
          e[r] += w[3 * r] * pp[0] + w[3 * r + 1] * pp[1] + w[3 * r + 2] * pp[2];
        }
      }
      for (int o = rec.x;;) {
        double u[2];
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          u[a] = 0.0;
#pragma unroll
          for (int r = 0; r < 6; ++r) u[a] += jac[9 * a + r] * c[r];
#pragma unroll
          for (int k = 0; k < 3; ++k) u[a] += jac[9 * a + 6 + k] * pp[k];
        }
        const double m0 = jac[18] * u[0] + jac[19] * u[1], m1 = jac[19] * u[0] + jac[20] * u[1];
#pragma unroll
        for (int r = 0; r < 6; ++r) e[r] += jac[r] * m0 + jac[9 + r] * m1;
#pragma unroll
        for (int k = 0; k < 3; ++k) s[k] += jac[6 + k] * m0 + jac[15 + k] * m1;
        if (++o >= rec.y) break;
#pragma unroll
        for (int k = 0; k < 21; ++k) jac[k] = A.jac[static_cast<int64_t>(k) * A.obs + o];
      }
      if (cf) {
#pragma unroll
        for (int r = 0; r < 6; ++r) atomicAdd(&sPose[6 * q.key_frame + r], e[r]);
      }
      for (int k = 0; k < 3; ++k) sPair[3 * tid + k] = s[k];
    }
    __syncthreads();
    if (point) {
      const int qa = b.point_pair[i] - T.pair_begin, qe = min(b.point_pair[i + 1] - T.pair_begin, kBlock);
      double v[6], y[3];
      for (int k = 0; k < 6; ++k) v[k] = A.vh[static_cast<int64_t>(k) * npf + i];
      y[0] = v[0] * p[0] + v[1] * p[1] + v[3] * p[2];
      y[1] = v[1] * p[0] + v[2] * p[1] + v[4] * p[2];
      y[2] = v[3] * p[0] + v[4] * p[1] + v[5] * p[2];
      for (int q2 = qa; q2 < qe; ++q2)
        for (int k = 0; k < 3; ++k) y[k] += sPair[3 * q2 + k];
      for (int k = 0; k < 3; ++k) {
        A.y[n6 + 3 * i + k] = y[k];
        py += p[k] * y[k];
      }
    }
    // No barrier here: the next tile writes sP, last read before this tile's second barrier, and sPair only after its
    // own first barrier, which every thread reaches after its reads of this one.
  }
  __syncthreads();
  for (int k = tid; k < n6; k += kBlock) {
    A.part[static_cast<int64_t>(blockIdx.x) * n6 + k] = sPose[k];
    py += sPc[k] * sPose[k];
    if (blockIdx.x == 0) {  // the key frames' own blocks
      const int j = k / 6;
      double s = 0.0;
      for (int c = 0; c < 6; ++c) s += A.uh[6 * k + c] * sPc[6 * j + c];
      py += sPc[k] * s;
    }
  }
  py = block_sum(py, sh);
  if (tid == 0) A.s_py[blockIdx.x] = py;
}

// The points' part of x += alpha p, r -= alpha y (INIT: x = 0, r = g), |r|^2, and the Schur right-hand side's share
// -sum W_G V*^-1 r. Workgroup g also adds the key-frame sums of k_adj_hvp for entries g, g + slots, ... into y.
template <bool INIT>
__global__ __launch_bounds__(kBlock) void k_adj_update(Batch b, AdjData A) {
  __shared__ double sPose[6 * kMaxFreePoses];
  __shared__ double sT[3 * kBlock];
  __shared__ double sh[4];
  if (!INIT && *A.done) return;
  const WindowDesc W = b.win[0];
  const int tid = threadIdx.x, ncf = W.ncf, npf = W.npf, n6 = A.n6;
  double alpha = 0.0;
  if (!INIT) {
    const double py = slot_sum(A.s_py, A.slots, sh);
    // negative or zero curvature along p: the Hessian is not positive definite here; stop with the current x
    // (truncated conjugate gradients, as in Steihaug's method; k_adj_reduced sets the flag)
    if (!(py > 0.0)) return;
    alpha = A.sc[4 + A.parity] / py;
    for (int k = blockIdx.x; k < n6; k += A.slots) {
      double s = 0.0;
      for (int g = tid; g < A.slots; g += kBlock) s += A.part[static_cast<int64_t>(g) * n6 + k];
      s = block_sum(s, sh);
      if (tid == 0) A.y[k] = s;
    }
  }
  for (int k = tid; k < n6; k += kBlock) sPose[k] = 0.0;
  double rr = 0.0;
  const int t0 = (A.tiles * blockIdx.x) / A.slots, t1 = (A.tiles * (blockIdx.x + 1)) / A.slots;
  for (int t = t0; t < t1; ++t) {
    const Tile T = b.btiles[t];
    const PairOf q = pair_of(b, T, npf, ncf);
    double w[18];
    if (q.coupled) {
#pragma unroll
      for (int k = 0; k < 18; ++k) w[k] = A.wg[static_cast<int64_t>(k) * A.pairs + q.pair];
    }
    const int i = T.point_begin + tid;
    if (i < T.point_end && i < npf) {
      double r[3], v[3];
      for (int k = 0; k < 3; ++k) {
        const int at = n6 + 3 * i + k;
        if (INIT) {
          A.x[at] = 0.0;
          r[k] = A.gd[at];
        } else {
          A.x[at] += alpha * A.p[at];
          r[k] = A.r[at] - alpha * A.y[at];
        }
        A.r[at] = r[k];
        rr += r[k] * r[k];
      }
      apply_vinv(b, i, r, v);
      for (int k = 0; k < 3; ++k) sT[3 * tid + k] = v[k];
    }
    __syncthreads();
    if (q.coupled) {
      const double* v = sT + 3 * q.point;
#pragma unroll
      for (int r = 0; r < 6; ++r)
        atomicAdd(&sPose[6 * q.key_frame + r], -(w[3 * r] * v[0] + w[3 * r + 1] * v[1] + w[3 * r + 2] * v[2]));
    }
    __syncthreads();
  }
  __syncthreads();
  for (int k = tid; k < n6; k += kBlock) A.part2[static_cast<int64_t>(blockIdx.x) * n6 + k] = sPose[k];
  rr = block_sum(rr, sh);
  if (tid == 0) A.s_rr[blockIdx.x] = rr;
}

// The key-frame part in one workgroup: x, r, |r|^2 and the convergence test, then z_c = S^-1 (r_c - sum W_G V*^-1 r) / 2
// with the dense inverse of the reduced system, and its share of r.z. 1024 threads: the Schur right-hand side's slots
// are added by row groups of threads, the product with the inverse by one wavefront per row.
template <bool INIT>
__global__ __launch_bounds__(1024) void k_adj_reduced(AdjData A) {
  __shared__ double red[1024], ec[6 * kMaxFreePoses], rc[6 * kMaxFreePoses], zs[6 * kMaxFreePoses];
  __shared__ double sh[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n6 = A.n6;
  if (!INIT && *A.done) return;
  auto wave_sums = [&](double x) {  // to sh, one per wavefront
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
    __syncthreads();
    if (lane == 0) sh[wave] = x;
    __syncthreads();
  };
  auto sum = [&](double x) {  // over the workgroup, fixed order
    wave_sums(x);
    double s = 0.0;
    for (int k = 0; k < 16; ++k) s += sh[k];
    return s;
  };
  // slots of the Schur right-hand side: entry k by the threads (row group h, k), eight loads in flight
  const int groups = n6 > 0 ? 1024 / n6 : 0, h = n6 > 0 ? tid / n6 : 0, k = n6 > 0 ? tid % n6 : 0;
  double e = 0.0;
  if (h < groups) {
    int g = h;
    double a[8] = {};
    for (; g + 7 * groups < A.slots; g += 8 * groups) {
#pragma unroll
      for (int u = 0; u < 8; ++u) a[u] += A.part2[static_cast<int64_t>(g + u * groups) * n6 + k];
    }
    for (; g < A.slots; g += groups) a[0] += A.part2[static_cast<int64_t>(g) * n6 + k];
    e = ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
  }
  red[tid] = e;
  double alpha = 0.0;
  if (!INIT) {
    // p.y in slot_sum's order, so that this step and its stop are those of k_adj_update to the last bit
    static_assert(kAdjSlots <= kBlock && kBlock == 256, "one slot per thread of four wavefronts");
    wave_sums(tid < A.slots ? A.s_py[tid] : 0.0);
    const double py = (sh[0] + sh[1]) + (sh[2] + sh[3]);
    if (!(py > 0.0)) {  // workgroup-uniform
      if (tid == 0) *A.done = 1;
      return;
    }
    alpha = A.sc[4 + A.parity] / py;
  }
  double rr = 0.0;
  for (int g = tid; g < A.slots; g += 1024) rr += A.s_rr[g];
  if (tid < n6) {
    double r;
    if (INIT) {
      A.x[tid] = 0.0;
      r = A.gd[tid];
    } else {
      const double* pc = A.pc + 6 * kMaxFreePoses * A.parity;
      const int j = tid / 6;
      double y = A.y[tid];
      for (int c = 0; c < 6; ++c) y += A.uh[6 * tid + c] * pc[6 * j + c];
      A.x[tid] += alpha * pc[tid];
      r = A.r[tid] - alpha * y;
    }
    A.r[tid] = r;
    rc[tid] = r;
    rr += r * r;
  }
  rr = sum(rr);  // its barriers also publish red and rc
  if (tid == 0) {
    bool stop;
    if (INIT) {
      A.sc[0] = rr;
      A.sc[2] = 0.0;
      stop = rr == 0.0;
    } else {
      A.sc[1] = rr;
      A.sc[2] += 1.0;
      stop = sqrt(rr / A.sc[0]) < A.tol;
    }
    if (stop) *A.done = 1;
  }
  if (tid < n6) {
    double v = rc[tid];
    for (int g = 0; g < groups; ++g) v += red[g * n6 + tid];
    ec[tid] = v;
  }
  __syncthreads();
  for (int i = wave; i < n6; i += 16) {
    const double* row = A.sinv + static_cast<int64_t>(i) * n6;
    double s = 0.0;
    for (int c = lane; c < n6; c += 64) s += row[c] * ec[c];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (lane == 0) {
      zs[i] = s;
      A.zc[i] = s;
      A.z[i] = 0.5 * s;
    }
  }
  __syncthreads();
  const double rz = sum(tid < n6 ? 0.5 * zs[tid] * rc[tid] : 0.0);
  if (tid == 0) A.sc[3] = rz;
}

// The points' part of z = M^-1 r: z_p = V*^-1 (r_p - sum W_G^T z_c) / 2 (M is twice the Gauss-Newton system), and its
// share of r.z. INIT: the first application, which also gives the Gauss-Newton step (z = 0 for a zero gradient).
template <bool INIT>
__global__ __launch_bounds__(kBlock) void k_adj_precond(Batch b, AdjData A) {
  __shared__ double sZc[6 * kMaxFreePoses];
  __shared__ double sPair[3 * kBlock];
  __shared__ double sh[4];
  if (!INIT && *A.done) return;
  const WindowDesc W = b.win[0];
  const int tid = threadIdx.x, ncf = W.ncf, npf = W.npf, n6 = A.n6;
  for (int k = tid; k < n6; k += kBlock) sZc[k] = A.zc[k];
  double rz = 0.0;
  const int t0 = (A.tiles * blockIdx.x) / A.slots, t1 = (A.tiles * (blockIdx.x + 1)) / A.slots;
  for (int t = t0; t < t1; ++t) {
    const Tile T = b.btiles[t];
    const PairOf q = pair_of(b, T, npf, ncf);
    double w[18];
    if (q.coupled) {
#pragma unroll
      for (int k = 0; k < 18; ++k) w[k] = A.wg[static_cast<int64_t>(k) * A.pairs + q.pair];
    }
    __syncthreads();  // sZc written; the previous tile's sPair is free
    if (q.valid) {
      double s[3] = {};
      if (q.coupled) {
        const double* c = sZc + 6 * q.key_frame;
#pragma unroll
        for (int r = 0; r < 6; ++r)
#pragma unroll
          for (int k = 0; k < 3; ++k) s[k] += w[3 * r + k] * c[r];
      }
      for (int k = 0; k < 3; ++k) sPair[3 * tid + k] = s[k];
    }
    __syncthreads();
    const int i = T.point_begin + tid;
    if (i < T.point_end && i < npf) {
      const int qa = b.point_pair[i] - T.pair_begin, qe = min(b.point_pair[i + 1] - T.pair_begin, kBlock);
      double r[3], d[3], z[3];
      for (int k = 0; k < 3; ++k) d[k] = r[k] = A.r[n6 + 3 * i + k];
      for (int q2 = qa; q2 < qe; ++q2)
        for (int k = 0; k < 3; ++k) d[k] -= sPair[3 * q2 + k];
      apply_vinv(b, i, d, z);
      for (int k = 0; k < 3; ++k) {
        z[k] *= 0.5;
        A.z[n6 + 3 * i + k] = z[k];
        rz += r[k] * z[k];
      }
    }
  }
  rz = block_sum(rz, sh);
  if (tid == 0) A.s_rz[blockIdx.x] = rz;
}

namespace {
__device__ __forceinline__ int64_t pk2(int i, int j) { return static_cast<int64_t>(i) * (i + 1) / 2 + j; }
}  // namespace

// L^-1 of the stored FP64 factor (packed lower L, then 1 / L_ii), dense row-major n x n (zero above the diagonal),
// one wavefront per column j: x = L^-1 e_j by forward substitution, each row's dot product over the lanes with a
// fixed butterfly. Run once per factored solution; the preconditioner then applies S^-1 = L^-T L^-1 as two
// parallel products instead of two serial triangular solves.
__global__ __launch_bounds__(64) void k_adj_linv(const double* Lst, int n, double* Linv) {
  __shared__ double x[256];
  const int j = blockIdx.x, lane = threadIdx.x;
  const double* idg = Lst + static_cast<int64_t>(n) * (n + 1) / 2;
  for (int i = lane; i < n; i += 64) x[i] = 0.0;
  sba_tiles::wave_lds_sync();
  for (int i = j; i < n; ++i) {
    double sum = 0.0;
    for (int k = j + lane; k < i; k += 64) sum += Lst[pk2(i, k)] * x[k];
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    if (lane == 0) x[i] = ((i == j ? 1.0 : 0.0) - sum) * idg[i];
    sba_tiles::wave_lds_sync();
  }
  for (int i = lane; i < n; i += 64) Linv[static_cast<int64_t>(i) * n + j] = i >= j ? x[i] : 0.0;
}

// S^-1 = L^-T L^-1 (dense, symmetric) from the inverse factor, one workgroup per row.
__global__ __launch_bounds__(kBlock) void k_adj_sinv(const double* Linv, int n, double* sinv) {
  const int i = blockIdx.x;
  for (int j = threadIdx.x; j < n; j += kBlock) {
    double s = 0.0;
#pragma unroll 4
    for (int k = max(i, j); k < n; ++k) s += Linv[static_cast<int64_t>(k) * n + i] * Linv[static_cast<int64_t>(k) * n + j];
    sinv[static_cast<int64_t>(i) * n + j] = s;
  }
}

// FP64 state of window 0 from its FP32 state (op 0; free rotations projected onto the rotation group), or a Newton step x <- x - a applied to it (op 1):
// T_j <- Exp(-a_j) T_j for the free key frames (math/twist.cpp:23-41 in FP64), p_i <- p_i - a_i for the free points.
__global__ __launch_bounds__(256) void k_adj_state(Batch b, double* spts, double* sposes, const double* a, int op) {
  const WindowDesc W = b.win[0];
  const int cur = b.st[0].cur;
  const float4* pts = cur ? b.pts1 : b.pts0;
  const float4* poses = cur ? b.poses1 : b.poses0;
  const int n6 = 6 * W.ncf;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < W.np; i += gridDim.x * blockDim.x) {
    if (op == 0) {
      const float4 q = pts[i];
      spts[3 * i] = q.x;
      spts[3 * i + 1] = q.y;
      spts[3 * i + 2] = q.z;
    } else if (i < W.npf) {
      for (int k = 0; k < 3; ++k) spts[3 * i + k] -= a[n6 + 3 * i + k];
    }
  }
  for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < W.nc; j += gridDim.x * blockDim.x) {
    double* T = sposes + 12 * j;
    if (op == 0) {
      double X[3][3];
      for (int r = 0; r < 3; ++r) {
        const float4 q = poses[3 * j + r];
        X[r][0] = q.x;
        X[r][1] = q.y;
        X[r][2] = q.z;
        T[4 * r + 3] = q.w;
      }
      // the FP32 rotations of the free key frames are orthonormal only to FP32 rounding; the Newton steps move
      // along Exp(xi) R and would otherwise settle on that orbit instead of the rotation group
      if (j < W.ncf) polar3(X);
      for (int r = 0; r < 3; ++r)
        for (int q = 0; q < 3; ++q) T[4 * r + q] = X[r][q];
    } else if (j < W.ncf) {
      const double w0 = -a[6 * j], w1 = -a[6 * j + 1], w2 = -a[6 * j + 2];
      const double v[3] = {-a[6 * j + 3], -a[6 * j + 4], -a[6 * j + 5]};
      const double theta = fmax(sqrt(w0 * w0 + w1 * w1 + w2 * w2), static_cast<double>(1.1920928955078125e-7f));
      const double c = cos(theta), st = sin(theta) / theta;
      const double n[3] = {w0 / theta, w1 / theta, w2 / theta};
      const double K[3][3] = {{c, -w2 * st, w1 * st}, {w2 * st, c, -w0 * st}, {-w1 * st, w0 * st, c}};
      double E[3][3];
      for (int r = 0; r < 3; ++r)
        for (int q = 0; q < 3; ++q) E[r][q] = K[r][q] + (1.0 - c) * n[r] * n[q];
      const double nxv[3] = {n[1] * v[2] - n[2] * v[1], n[2] * v[0] - n[0] * v[2], n[0] * v[1] - n[1] * v[0]};
      const double nnv[3] = {n[1] * nxv[2] - n[2] * nxv[1], n[2] * nxv[0] - n[0] * nxv[2], n[0] * nxv[1] - n[1] * nxv[0]};
      double et[3];
      for (int r = 0; r < 3; ++r) et[r] = v[r] + ((1.0 - c) / theta * nxv[r] + (1.0 - st) * nnv[r]);
      double R[3][4];
      for (int r = 0; r < 3; ++r)
        for (int q = 0; q < 4; ++q) R[r][q] = T[4 * r + q];
      for (int r = 0; r < 3; ++r) {
        for (int q = 0; q < 3; ++q) T[4 * r + q] = E[r][0] * R[0][q] + E[r][1] * R[1][q] + E[r][2] * R[2][q];
        T[4 * r + 3] = E[r][0] * R[0][3] + E[r][1] * R[1][3] + E[r][2] * R[2][3] + et[r];
      }
    }
  }
}

namespace sba_dev {

hipError_t launch_adj_state(const Batch& b, double* spts, double* sposes, const double* a, int op, hipStream_t s) {
  hipLaunchKernelGGL(k_adj_state, dim3(64), dim3(256), 0, s, b, spts, sposes, a, op);
  return hipGetLastError();
}

hipError_t launch_adj_assemble(const Batch& b, const AdjData& A, bool hess, hipStream_t s) {
  if (hess)
    hipLaunchKernelGGL(k_adj_assemble<true>, dim3(A.slots), dim3(kBlock), 0, s, b, A);
  else
    hipLaunchKernelGGL(k_adj_assemble<false>, dim3(A.slots), dim3(kBlock), 0, s, b, A);
  if (A.n6 > 0) hipLaunchKernelGGL(k_adj_gather, dim3(27 * (A.n6 / 6)), dim3(kBlock), 0, s, b, A, hess ? 1 : 0);
  return hipGetLastError();
}

hipError_t launch_adj_start(const Batch& b, const AdjData& A, hipStream_t s) {
  hipLaunchKernelGGL(k_adj_update<true>, dim3(A.slots), dim3(kBlock), 0, s, b, A);
  hipLaunchKernelGGL(k_adj_reduced<true>, dim3(1), dim3(1024), 0, s, A);
  hipLaunchKernelGGL(k_adj_precond<true>, dim3(A.slots), dim3(kBlock), 0, s, b, A);
  return hipGetLastError();
}

hipError_t launch_adj_iteration(const Batch& b, AdjData A, int it, hipStream_t s) {
  A.parity = it & 1;
  hipLaunchKernelGGL(k_adj_hvp, dim3(A.slots), dim3(kBlock), 0, s, b, A, it);
  hipLaunchKernelGGL(k_adj_update<false>, dim3(A.slots), dim3(kBlock), 0, s, b, A);
  hipLaunchKernelGGL(k_adj_reduced<false>, dim3(1), dim3(1024), 0, s, A);
  hipLaunchKernelGGL(k_adj_precond<false>, dim3(A.slots), dim3(kBlock), 0, s, b, A);
  return hipGetLastError();
}

hipError_t launch_adj_obs_grad(const Batch& b, const AdjData& A, const int32_t* orig, hipStream_t s) {
  if (A.tiles > 0) hipLaunchKernelGGL(k_adj_obs_grad, dim3(A.tiles), dim3(kBlock), 0, s, b, A, orig);
  return hipGetLastError();
}

// The dense inverse of the reduced system from the stored factor (n <= 240), through its inverse factor.
hipError_t launch_adj_inverse(const double* Lst, int n, double* Linv, double* sinv, hipStream_t s) {
  if (n > 6 * kMaxFreePoses) return hipErrorInvalidValue;
  if (n > 0) {
    hipLaunchKernelGGL(k_adj_linv, dim3(n), dim3(64), 0, s, Lst, n, Linv);
    hipLaunchKernelGGL(k_adj_sinv, dim3(n), dim3(kBlock), 0, s, Linv, n, sinv);
  }
  return hipGetLastError();
}

}  // namespace sba_dev
