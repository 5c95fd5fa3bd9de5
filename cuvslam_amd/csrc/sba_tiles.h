// Device helpers shared by the FP64 factor kernels: 16 x 16 FP64 tiles in the matrix-core layout
// (v_mfma_f64_16x16x4_f64: element (4v + lane/16, lane%16) in register v of the lane, i.e. 64 v + lane in
// row-major order), their trailing update, the one-wavefront Cholesky of a diagonal tile, and lane reductions.
#pragma once

#include <hip/hip_runtime.h>

#include <stdint.h>

namespace sba_tiles {

// Makes the LDS writes of some lanes of a wavefront visible to the later LDS reads of the other lanes: without
// it the compiler may satisfy a lane's read before the stores that only other lanes execute.
__device__ __forceinline__ void wave_lds_sync() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_wave_barrier();
  asm volatile("" ::: "memory");
}

typedef double double4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ double readlane_d(double x, int lane) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(x), lane);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(x), lane);
  return __hiloint2double(hi, lo);
}


__device__ __forceinline__ double4v mfma64(double a, double b, double4v c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// c - P_J^T P_I for two 16 x 16 row-major tiles in LDS (A operand lane l: P_J[4q + l/16][l%16] = 64 q + l)
__device__ __forceinline__ double4v tile_update(double4v c, const double* pj, const double* pi, int lane) {
#pragma unroll
  for (int q = 0; q < 4; ++q) c = mfma64(-pj[64 * q + lane], pi[64 * q + lane], c);
  return c;
}

// A wavefront-uniform value the compiler may not hoist out of the enclosing loop: keeps the per-tile LDS
// addresses from being precomputed for every tile slot at once (which would cost a register per slot).
__device__ __forceinline__ int in_loop(int x) {
  asm volatile("" : "+s"(x));
  return x;
}

__device__ __forceinline__ double sum_rows4(double x) {  // over lanes l, l^16, l^32, l^48
  x += __shfl_xor(x, 16);
  x += __shfl_xor(x, 32);
  return x;
}

__device__ __forceinline__ double sum_row16(double x) {  // over the 16 lanes of l's row group
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) x += __shfl_xor(x, o);
  return x;
}

// An estimate e of 1/sqrt(d) refined by a third-order step (the series of (1 - h)^-1/2 with h = 1 - d e^2: the cube of
// the hardware estimate's error is below rounding, its square is not always), and 1/sqrt(d) from that estimate.
__device__ __forceinline__ double refine_rsqrt(double d, double e) {
  const double h = 1.0 - d * e * e;
  return e + e * h * (0.5 + 0.375 * h);
}
__device__ __forceinline__ double rsqrt1(double d) { return refine_rsqrt(d, __builtin_amdgcn_rsq(d)); }

// Cholesky A = U^T U of a symmetric 16 x 16 tile held by one wavefront in the FP64 matrix-core layout (cell
// (4v + lane/16, lane%16) in t[v]) together with X = U^-T, as one elimination of [A | I] by panels of four rows.
// Register v of the layout is exactly the panel of rows 4v..4v+3, and it is at once the B operand of a 4 x 16 factor
// and the A operand of its transpose, so a panel step needs no data movement:
//   the 4 x 4 diagonal block is broadcast with readlane, factored and inverted by every lane (M = L_vv^-1);
//   U_v = M A_v and X_v = M I_v, one matrix instruction each; A -= U_v^T U_v and I -= U_v^T X_v, one each.
// On return t holds U (zero below the diagonal), X^T is written to xt (row-major) and 1 / U_ii to rdiag. False on a
// non-positive pivot (the values are then dropped by the callers).
//
// A serial chain bounds it: four 4 x 4 factors (a reciprocal square root and a few dependent FMAs per pivot) and two
// dependent matrix instructions each. Measured alone on one wavefront: 2.67 us with a column-by-column factorization
// and a forward substitution for X through LDS, 1.90 us as a column-by-column elimination of [A | I], 1.72 us in this
// form; the reconstruction error of a random tile fell from 9e-16 to 7e-16, that of X from 8e-16 to 3e-16.
__device__ inline bool factor_tile(double4v& t, double* xt, double* rdiag, int lane) {
  const int row = lane >> 4, col = lane & 15;
  double4v x, u;
#pragma unroll
  for (int v = 0; v < 4; ++v) x[v] = 4 * v + row == col ? 1.0 : 0.0;
  bool ok = true;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    // entry (r, c), r <= c, of the diagonal block
    auto at = [&](int r, int c) { return readlane_d(t[v], 16 * r + 4 * v + c); };
    const double a00 = at(0, 0), a01 = at(0, 1), a11 = at(1, 1), a02 = at(0, 2), a12 = at(1, 2), a03 = at(0, 3),
                 a13 = at(1, 3), a22 = at(2, 2), a23 = at(2, 3), a33 = at(3, 3);
    // Pivots in pairs: the second of a pair is det / first, so the estimates of both reciprocal square roots start
    // together; the second is then refined against the pivot itself, which keeps the accuracy of the plain recurrence.
    const double i0 = rsqrt1(a00), f1 = __builtin_amdgcn_rsq(a00 * a11 - a01 * a01) * a00;
    const double l10 = a01 * i0, l20 = a02 * i0, l30 = a03 * i0;
    const double d1 = a11 - l10 * l10, i1 = refine_rsqrt(d1, f1 * i0);
    const double l21 = (a12 - l10 * l20) * i1, l31 = (a13 - l10 * l30) * i1;
    const double d2 = (a22 - l20 * l20) - l21 * l21, b23 = (a23 - l20 * l30) - l21 * l31,
                 b33 = (a33 - l30 * l30) - l31 * l31;
    const double i2 = rsqrt1(d2), f3 = __builtin_amdgcn_rsq(d2 * b33 - b23 * b23) * d2;
    const double l32 = b23 * i2;
    const double d3 = b33 - l32 * l32, i3 = refine_rsqrt(d3, f3 * i2);
    ok = ok && a00 > 0.0 && d1 > 0.0 && d2 > 0.0 && d3 > 0.0;
    // M = L_vv^-1 as the A operand: lane l holds M[l % 16][l / 16], rows past the fourth zero
    const double m10 = -(l10 * i0) * i1;
    const double q20 = l20 * i0 + l21 * m10, q21 = l21 * i1, q30 = l30 * i0 + l31 * m10, q31 = l31 * i1;
    const double m20 = -q20 * i2, m21 = -q21 * i2;
    double m = lane == 0 ? i0 : 0.0;
    m = lane == 1 ? m10 : m;
    m = lane == 17 ? i1 : m;
    m = lane == 2 ? m20 : m;
    m = lane == 18 ? m21 : m;
    m = lane == 34 ? i2 : m;
    m = lane == 35 ? -(l32 * i2) * i3 : m;
    m = lane == 3 ? -(q30 + l32 * m20) * i3 : m;
    m = lane == 19 ? -(q31 + l32 * m21) * i3 : m;
    m = lane == 51 ? i3 : m;
    const double4v zero = {0.0, 0.0, 0.0, 0.0};
    const double uv = mfma64(m, t[v], zero)[0];
    // The next panel waits for A only, so its product goes first. Rows up to this panel are final in u and x and
    // columns up to it are eliminated: what the products leave there is not read again.
    if (v < 3) t = mfma64(-uv, uv, t);
    const double xv = mfma64(m, x[v], zero)[0];
    if (v < 3) {
      const double4v xn = mfma64(-uv, xv, x);
#pragma unroll
      for (int w = v + 1; w < 4; ++w) x[w] = xn[w];
    }
    u[v] = 4 * v + row <= col ? uv : 0.0;
    x[v] = xv;
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    t[v] = u[v];
    xt[16 * col + 4 * v + row] = x[v];
    if (4 * v + row == col) rdiag[col] = x[v];
  }
  return ok;
}

// Sum over the 16 lanes of each row of 16 (DPP within rows; every lane gets its row's sum).
__device__ __forceinline__ double dpp_f64(double x, int ctrl_sel) {
  int lo = __double2loint(x), hi = __double2hiint(x);
  switch (ctrl_sel) {
    case 0:
      lo = __builtin_amdgcn_update_dpp(0, lo, 0xB1, 0xF, 0xF, false);  // quad_perm [1,0,3,2]
      hi = __builtin_amdgcn_update_dpp(0, hi, 0xB1, 0xF, 0xF, false);
      break;
    case 1:
      lo = __builtin_amdgcn_update_dpp(0, lo, 0x4E, 0xF, 0xF, false);  // quad_perm [2,3,0,1]
      hi = __builtin_amdgcn_update_dpp(0, hi, 0x4E, 0xF, 0xF, false);
      break;
    case 2:
      lo = __builtin_amdgcn_update_dpp(0, lo, 0x124, 0xF, 0xF, false);  // row_ror:4
      hi = __builtin_amdgcn_update_dpp(0, hi, 0x124, 0xF, 0xF, false);
      break;
    default:
      lo = __builtin_amdgcn_update_dpp(0, lo, 0x128, 0xF, 0xF, false);  // row_ror:8
      hi = __builtin_amdgcn_update_dpp(0, hi, 0x128, 0xF, 0xF, false);
      break;
  }
  return __hiloint2double(hi, lo);
}

__device__ __forceinline__ double sum_row16_dpp(double x) {
  x += dpp_f64(x, 0);
  x += dpp_f64(x, 1);
  x += dpp_f64(x, 2);
  x += dpp_f64(x, 3);
  return x;
}

}  // namespace sba_tiles
