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

// 1/sqrt(d) of a normal positive d: the hardware estimate e refined by a third-order step (the series of (1 - h)^-1/2
// with h = 1 - d e^2: the cube of the estimate's error is below rounding, its square is not always). Not a number for
// every other d, zero and infinity included.
__device__ __forceinline__ double rsqrt1(double d) {
  const double e = __builtin_amdgcn_rsq(d), h = 1.0 - d * e * e;
  return e + e * h * (0.5 + 0.375 * h);
}

// r[k] = x of the lane of the same column (lane % 16) in row k (lanes 16 k .. 16 k + 15), in every lane.
__device__ __forceinline__ void rows_of(double x, double (&r)[4]) {
  auto half = [](unsigned w, unsigned (&o)[4]) {
    const auto a = __builtin_amdgcn_permlane32_swap(w, w, false, false);      // rows 0 1 0 1 and 2 3 2 3
    const auto b = __builtin_amdgcn_permlane16_swap(a[0], a[0], false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(a[1], a[1], false, false);
    o[0] = b[0];
    o[1] = b[1];
    o[2] = c[0];
    o[3] = c[1];
  };
  unsigned lo[4], hi[4];
  half(__double2loint(x), lo);
  half(__double2hiint(x), hi);
#pragma unroll
  for (int k = 0; k < 4; ++k) r[k] = __hiloint2double(hi[k], lo[k]);
}

// Cholesky A = U^T U of a symmetric 16 x 16 tile held by one wavefront in the FP64 matrix-core layout (cell
// (4v + lane/16, lane%16) in t[v]) together with X = U^-T, as one elimination of [A | I] by panels of four rows.
// Register v of the layout is exactly the panel of rows 4v..4v+3:
//   the 4 x 4 diagonal block is broadcast with readlane and factored by every lane (the plain recurrence, L_vv);
//   U_v = L_vv^-1 A_v and X_v = L_vv^-1 I_v by forward substitution, every lane with its column's four rows;
//   A -= U_v^T U_v and I -= U_v^T X_v, one matrix instruction each: the panel is at once the B operand and the A operand
//   of its transpose.
// On return t holds U (zero below the diagonal), X^T is written to xt (row-major) and, unless rdiag is null, 1 / U_ii to
// rdiag. False on a pivot that is not positive and finite (the values are then dropped by the callers).
//
// A serial chain bounds it: 16 reciprocal square roots with a few dependent FMAs each, and one matrix instruction per
// panel between them; the substitutions run beside the chain of their own block. Measured alone on one wavefront: 1.07 us;
// 1.32 us with the rows as products with the explicit inverse of L_vv and every second square root started from a 2 x 2
// determinant; 1.80 us as a column-by-column factorization with X formed through LDS. Backward stable: over 2000 tiles
// each with second pivots of a relative size of 1 to 1e-15, |U^T U - A| stays within 9e-16 of sqrt(a_ii a_jj) and
// |U^T X - I| within 3.3e-16 of |U^T| |X| (6e-15 and 8e-15 column by column; with the explicit inverse both grew with
// the block's condition, to 1e-10 and 1e-4 at 1e-12, and a determinant that cancelled to zero gave infinities that
// passed as a good factor).
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
    const double i0 = rsqrt1(a00), l10 = a01 * i0, l20 = a02 * i0, l30 = a03 * i0;
    const double i1 = rsqrt1(a11 - l10 * l10);
    const double l21 = (a12 - l10 * l20) * i1, l31 = (a13 - l10 * l30) * i1;
    const double i2 = rsqrt1((a22 - l20 * l20) - l21 * l21);
    const double l32 = ((a23 - l20 * l30) - l21 * l31) * i2;
    const double i3 = rsqrt1(((a33 - l30 * l30) - l31 * l31) - l32 * l32);
    ok = ok && i0 > 0.0 && i1 > 0.0 && i2 > 0.0 && i3 > 0.0;
    auto solve = [&](double b) {  // this lane's entry of L_vv^-1 b
      double r[4];
      rows_of(b, r);
      r[0] *= i0;
      r[1] = (r[1] - l10 * r[0]) * i1;
      r[2] = ((r[2] - l20 * r[0]) - l21 * r[1]) * i2;
      r[3] = (((r[3] - l30 * r[0]) - l31 * r[1]) - l32 * r[2]) * i3;
      return row < 2 ? (row == 0 ? r[0] : r[1]) : (row == 2 ? r[2] : r[3]);
    };
    const double uv = solve(t[v]);
    // The next panel waits for A only, so its product goes first. Rows up to this panel are final in u and x and
    // columns up to it are eliminated: what the products leave there is not read again.
    if (v < 3) t = mfma64(-uv, uv, t);
    const double xv = solve(x[v]);
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
    if (rdiag && 4 * v + row == col) rdiag[col] = x[v];
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
