// Reduced camera system of windows with more than kMaxFreePoses free key frames ("mapped" windows, e.g. a large
// multi-camera map with a reduced system of order ~1200).
//
// The Schur kernel stages at most kMaxFreePoses free key frames per chunk; a mapped window's chunks carry the
// list of the free key frames they stage (chunk_map, increasing). Here:
//   k_gather      A = U + lambda diag(U) - sum Z Z^T in FP64 (dense, row-major lower triangle), rhs e: each
//                 key-frame block sums its contributions from the chunk records in chunk order (a plan built
//                 with the chunks), so the system, like the small windows' reduction, has fixed bits
//   k_lfirst / k_lstep   right-looking blocked Cholesky (Golub & Van Loan, Matrix Computations, Algorithm 4.2.10)
//                 with 64 x 64 blocks, one launch per block column: a diagonal block is factored, with its inverse, on
//                 the 16 x 16 FP64 tile scheme of the small-window factor; the panel below it is a product with that
//                 inverse, formed by the workgroups of the trailing update that need it; the workgroup of the next
//                 diagonal block goes on to factor it. The forward substitution L y = e rides along.
//   k_bsolve      L^T x = y by 64-row blocks with the kept inverses, in one workgroup; then the pose step, its
//                 max-norm and dc^T diag(U) dc, trial key frames
// A non-positive pivot clears the window's chol_ok; the later kernels then return, and the LM decision raises
// lambda (schur_complement_bundler_gpu.cpp:175-185), as for the small windows.
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>

#include "sba_device.h"
#include "sba_tiles.h"

using namespace sba_dev;
using namespace sba_tiles;

namespace {

constexpr int kLB = 64;        // block of the large factorization
constexpr int kGather = 8;     // contributions whose loads k_gather issues together
constexpr int kGatherWaves = 4;  // wavefronts of k_gather that share one key-frame block's contributions

struct Large {
  double* A;     // n x n, row-major; the lower triangle holds A; L^T replaces the blocks above the diagonal
  double* rhs;   // e, then y, then x
  double* du;    // diag(U)
  double* Linv;  // per 64-row block: the inverse of its diagonal block of L (64 x 64, row-major, lower)
  int n;
};

__device__ __forceinline__ Large large_of(const Batch& b, const WindowDesc& W) {
  const int n = 6 * W.ncf;
  double* A = b.A + W.a_off;
  const int64_t nn = static_cast<int64_t>(n) * n;
  return Large{A, A + nn, A + nn + n, A + nn + 2 * n, n};
}

}  // namespace

// A = U + lambda diag(U) - sum Z Z^T (lower triangle), rhs = e, du = diag(U); chol_ok set for the factor.
// One workgroup per key-frame block (a, b), a <= b (blockIdx.x enumerates the upper blocks row by row). Lane 6 r + c
// of each of the kGatherWaves wavefronts sums element (r, c) of the chunk-local block (la, lb) (36 contiguous
// floats of a record) in FP64 over its share of the block's contributions, in their listed (chunk) order; the
// shares' sums are added in wavefront order.
// A(6 b + c, 6 a + r) = -sum; in a diagonal block lanes with r <= c add U and lambda diag U, lanes 36..41 sum e
// and lanes 42..47 diag U. The sums do not depend on the order the hardware runs the chunks or the workgroups.
__global__ __launch_bounds__(64 * kGatherWaves) void k_gather(Batch b, int w) {
  __shared__ double red[3][kGatherWaves - 1][64];  // wavefronts 1..: their sums z, u, d
  const WindowDesc W = b.win[w];
  WindowState* St = b.st + w;
  if (St->done) return;
  const int ncf = W.ncf, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  // upper block t = blockIdx.x: row ka holds blocks ka..ncf-1, rows before it ka ncf - ka (ka - 1) / 2 blocks
  const int t = blockIdx.x;
  int ka = static_cast<int>((2.0 * ncf + 1.0 - sqrt((2.0 * ncf + 1.0) * (2.0 * ncf + 1.0) - 8.0 * t)) / 2.0);
  ka = max(0, min(ka, ncf - 1));
  while (ka > 0 && ka * ncf - (ka * (ka - 1)) / 2 > t) --ka;
  while (ka + 1 < ncf && (ka + 1) * ncf - ((ka + 1) * ka) / 2 <= t) ++ka;
  const int kb = ka + t - (ka * ncf - (ka * (ka - 1)) / 2);
  if (t == 0 && threadIdx.x == 0) St->chol_ok = 1;
  const Large L = large_of(b, W);
  const int n = L.n;
  const bool diag = ka == kb;
  const int r = lane / 6, c = lane % 6;
  // what this lane sums: 0 Z Z^T element (with U and diag U on the diagonal), 1 e, 2 diag U, -1 nothing
  int kind = -1;
  if (lane < 36 && (!diag || r <= c)) kind = 0;
  else if (diag && lane >= 36 && lane < 48) kind = lane < 42 ? 1 : 2;
  const int q = lane >= 36 ? (lane - 36) % 6 : 0;
  const int32_t* first = b.gfirst + W.gfirst_off + ka * ncf + kb;
  const int nall = first[1] - first[0];
  const int kbeg = first[0] + (nall * wave) / kGatherWaves, kend = first[0] + (nall * (wave + 1)) / kGatherWaves;
  const bool want_u = kind == 0 && diag, want_d = want_u && r == c;
  double z = 0.0, u = 0.0, d = 0.0;
  // kGather contributions at a time: their plan entries, then their record values, all loads of a batch in
  // flight together; the values are then added one after another in the plan's order
  for (int k0 = kbeg; kind >= 0 && k0 < kend; k0 += kGather) {
    int64_t oz[kGather], ou[kGather], od[kGather];
#pragma unroll
    for (int t = 0; t < kGather; ++t) {
      const int4 g = b.gcon[min(k0 + t, kend - 1)];
      const int64_t rec = (static_cast<int64_t>(g.w) << 32) | static_cast<uint32_t>(g.z);
      const int la = g.y & 255, lb = (g.y >> 8) & 255, nloc = g.y >> 24;
      const int64_t tail = rec + 36 * (nloc * (nloc + 1) / 2);
      if (kind == 0) {
        oz[t] = rec + 36 * (la * nloc - (la * (la - 1)) / 2 + (lb - la)) + 6 * r + c;
      } else {
        oz[t] = tail + (kind == 1 ? 21 : 27) * nloc + 6 * la + q;
      }
      ou[t] = tail + 21 * la + (want_u ? 6 * r - (r * (r - 1)) / 2 + (c - r) : 0);
      od[t] = tail + 27 * nloc + 6 * la + r;
    }
    float vz[kGather], vu[kGather], vd[kGather];
#pragma unroll
    for (int t = 0; t < kGather; ++t) {
      vz[t] = b.part[oz[t]];
      vu[t] = want_u ? b.part[ou[t]] : 0.f;
      vd[t] = want_d ? b.part[od[t]] : 0.f;
    }
#pragma unroll
    for (int t = 0; t < kGather; ++t)
      if (k0 + t < kend) {
        z += static_cast<double>(vz[t]);
        u += static_cast<double>(vu[t]);
        d += static_cast<double>(vd[t]);
      }
  }
  if (wave > 0) {
    red[0][wave - 1][lane] = z;
    red[1][wave - 1][lane] = u;
    red[2][wave - 1][lane] = d;
  }
  __syncthreads();
  if (wave > 0 || kind < 0) return;
#pragma unroll
  for (int v = 0; v < kGatherWaves - 1; ++v) {
    z += red[0][v][lane];
    u += red[1][v][lane];
    d += red[2][v][lane];
  }
  if (kind == 0) {
    double v = u - z;
    if (diag && r == c) v += static_cast<double>(St->lambda) * d;
    L.A[static_cast<int64_t>(6 * kb + c) * n + 6 * ka + r] = v;
  } else if (kind == 1) {
    L.rhs[6 * ka + q] = z;
  } else {
    L.du[6 * ka + q] = z;
  }
}

// Staged 64 x 64 operands: 16 x 16 tiles of kTs doubles with rows of kTr (one double of padding, so that the transposing
// writes of a wavefront fall into different banks). Tile (I, M) of P, at 4 I + M, holds element [m][i] =
// P[16 I + i][16 M + m], the operand layout of the matrix instructions (lane l reads [4q + l/16][l%16]).
constexpr int kTr = 17, kTs = 16 * kTr;

// 256 threads: each loads its 16 entries in one batch, then stores them.
__device__ __forceinline__ void stage_transposed(double* sT, const double* src, int64_t ld, int rows, int cols,
                                                 int tid) {
  constexpr int kPer = kLB * kLB / 256;
  double v[kPer];
#pragma unroll
  for (int it = 0; it < kPer; ++it) {
    const int idx = tid + 256 * it, r = idx / kLB, c = idx % kLB;  // row-major: consecutive threads, columns
    v[it] = (r < rows && c < cols) ? src[static_cast<int64_t>(r) * ld + c] : 0.0;
  }
#pragma unroll
  for (int it = 0; it < kPer; ++it) {
    const int idx = tid + 256 * it, r = idx / kLB, c = idx % kLB;
    sT[kTs * (4 * (r >> 4) + (c >> 4)) + kTr * (c & 15) + (r & 15)] = v[it];
  }
}

// c - P Q^T of one tile of P and one of Q, both staged as above.
__device__ __forceinline__ double4v staged_update(double4v c, const double* p, const double* q, int at) {
#pragma unroll
  for (int s = 0; s < 4; ++s) c = mfma64(-p[4 * kTr * s + at], q[4 * kTr * s + at], c);
  return c;
}

// Shared memory of factor_block, in doubles: diagonal tiles, their inverses transposed, the current panel, the
// off-diagonal tiles of A and of X, the right-hand side.
constexpr int kFbDg = 0, kFbXT = kFbDg + 4 * 256, kFbP = kFbXT + 4 * 256, kFbU = kFbP + 4 * 256, kFbX = kFbU + 6 * 256,
              kFbVec = kFbX + 6 * 256, kFbY = kFbVec + kLB, kFbWords = kFbY + kLB;

// pair index of tile (J, I), J < I < 4: 0 (0,1) 1 (0,2) 2 (0,3) 3 (1,2) 4 (1,3) 5 (2,3)
__device__ __forceinline__ int pair_of(int J, int I) { return J == 0 ? I - 1 : (J == 1 ? I + 1 : 5); }

// Cholesky A = U^T U of a 64 x 64 block by one workgroup of 256 threads, with X = U^-T and y = X e. The block's upper
// tiles come in shared memory (sm + kFbDg, kFbU, row-major 16 x 16) and e in sm + kFbVec, with a barrier after them.
// Wavefront 0 factors the diagonal tiles one after another (factor_tile); wavefronts 1..3 hold the six off-diagonal
// tiles U_JI (J < I) and the six tiles X_IJ below the diagonal of the identity in registers and carry both along:
//   panel     U_KI = X_KK A_KI, e_I -= U_KI^T y_K;   X_KJ = X_KK E_KJ;
//   trailing  A_JI -= U_KJ^T U_KI;                   E_IJ -= U_KI^T X_KJ,
// on the FP64 matrix cores while wavefront 0 factors the next tile, so that the block's inverse is complete when its
// last tile is. False (in every thread) on a non-positive pivot; every thread runs the same barriers.
// On return X is written to Xg (64 x 64 row-major, zero above the diagonal) and y to rhs.
__device__ bool factor_block(double* sm, int* flag, double* Xg, double* rhs, int kb, int tid) {
  constexpr int T = kLB / 16;  // 4 tile columns
  double* sDg = sm + kFbDg;
  double* sXT = sm + kFbXT;
  double* sP = sm + kFbP;
  double* sU = sm + kFbU;
  double* sX = sm + kFbX;
  double *vec = sm + kFbVec, *ys = sm + kFbY;
  const int lane = tid & 63, li = lane >> 4, lj = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  auto forward = [&](int K) {  // y_K = X_KK e_K, lane l holds y_K[l % 16]
    const double* xt = sXT + 256 * K;
    double yk = 0.0;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) yk += xt[16 * (4 * li + kk) + lj] * vec[16 * K + 4 * li + kk];
    return sum_rows4(yk);
  };
  if (wave == 0) {
    for (int K = -1; K < T; ++K) {
      if (K >= 0 && *flag) break;  // at K = -1 no barrier lies between the read and a failed tile's write
      if (K >= 0) {
        const double yk = forward(K);
        if (lane < 16) ys[16 * K + lane] = yk;
        __syncthreads();
      }
      if (K + 1 < T) {
        double* tk = sDg + 256 * (K + 1);
        double4v dt;
#pragma unroll
        for (int v = 0; v < 4; ++v) dt[v] = tk[64 * v + lane];
        if (K >= 0) dt = tile_update(dt, sP + 256 * (K + 1), sP + 256 * (K + 1), lane);
        if (!factor_tile(dt, sXT + 256 * (K + 1), nullptr, lane) && lane == 0) *flag = 1;
      }
      __syncthreads();
    }
  } else {
    // two register tiles of U and of X per wavefront: pair index m = 3 s + wave - 1
    int tJ[2], tI[2];
    double4v acc[2], inv[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int m = 3 * s + wave - 1;
      tJ[s] = m < 3 ? 0 : (m < 5 ? 1 : 2);
      tI[s] = m < 3 ? m + 1 : (m < 5 ? m - 1 : 3);
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[s][v] = sU[256 * m + 64 * v + lane];
      inv[s] = double4v{0.0, 0.0, 0.0, 0.0};
    }
    for (int K = -1; K < T; ++K) {
      if (K >= 0 && *flag) break;
      if (K >= 0) {
        const double* xt = sXT + 256 * K;
        const double yk = forward(K);
        double yv[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) yv[v] = __shfl(yk, 4 * v + li);  // y_K[4v + lane/16]
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          if (tJ[s] == K || tI[s] == K) {
            // X_KK times a tile: the B operand of chunk q is register q of the tile
            const double4v in = tJ[s] == K ? acc[s] : inv[s];
            double4v u = double4v{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int q = 0; q < 4; ++q) u = mfma64(xt[64 * q + lane], in[q], u);
            double* dst = tJ[s] == K ? sP + 256 * tI[s] : sX + 256 * pair_of(tJ[s], K);
#pragma unroll
            for (int v = 0; v < 4; ++v) dst[64 * v + lane] = u[v];
            if (tJ[s] == K) {
              double p = 0.0;
#pragma unroll
              for (int v = 0; v < 4; ++v) p += u[v] * yv[v];
              p = sum_rows4(p);
              if (lane < 16) vec[16 * tI[s] + lane] -= p;
            }
          }
        }
        __syncthreads();
        // trailing: the diagonal tiles past K + 1 (LDS), then this wavefront's tiles
        for (int J = K + 1 + wave; J < T; J += 3) {
          double* tj = sDg + 256 * J;
          double4v t;
#pragma unroll
          for (int v = 0; v < 4; ++v) t[v] = tj[64 * v + lane];
          t = tile_update(t, sP + 256 * J, sP + 256 * J, lane);
#pragma unroll
          for (int v = 0; v < 4; ++v) tj[64 * v + lane] = t[v];
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          if (tJ[s] > K) {
            acc[s] = tile_update(acc[s], sP + 256 * tJ[s], sP + 256 * tI[s], lane);
          } else if (tI[s] > K) {
            // B operand X_KJ[4q + l/16][l%16]: X_KK from its transpose, the others row-major
            const double* U = sP + 256 * tI[s];
            const double* X = tJ[s] == K ? xt + 16 * lj + li : sX + 256 * pair_of(tJ[s], K) + lane;
            const int step = tJ[s] == K ? 4 : 64;
#pragma unroll
            for (int q = 0; q < 4; ++q) inv[s] = mfma64(-U[64 * q + lane], X[step * q], inv[s]);
          }
        }
      }
      __syncthreads();
    }
  }
  if (*flag) return false;
  for (int idx = tid; idx < kLB * kLB; idx += 256) {
    const int R = idx / kLB, Cc = idx % kLB;
    const int I = R >> 4, J = Cc >> 4, a = R & 15, c = Cc & 15;
    double x = 0.0;
    if (J == I) x = sXT[256 * I + 16 * c + a];
    else if (J < I) x = sX[256 * pair_of(J, I) + 16 * a + c];
    Xg[idx] = x;
  }
  if (tid < kb) rhs[tid] = ys[tid];
  return true;
}

// The first diagonal block: read, factored, its inverse and y_0 written.
__global__ __launch_bounds__(256) void k_lfirst(Batch b, int w) {
  __shared__ double sm[kFbWords];
  __shared__ int flag;
  const WindowDesc W = b.win[w];
  WindowState* St = b.st + w;
  if (St->done || !St->chol_ok) return;
  const Large L = large_of(b, W);
  const int n = L.n, kb = min(kLB, n), tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  // upper tiles (wave, I), read from the lower triangle; identity past the matrix
  for (int I = wave; I < 4; ++I) {
    double* dst = I == wave ? sm + kFbDg + 256 * I : sm + kFbU + 256 * pair_of(wave, I);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r = 16 * wave + 4 * v + (lane >> 4), c = 16 * I + (lane & 15);
      dst[64 * v + lane] = r < kb && c < kb ? L.A[static_cast<int64_t>(max(r, c)) * n + min(r, c)] : (r == c ? 1.0 : 0.0);
    }
  }
  if (tid < kLB) sm[kFbVec + tid] = tid < kb ? L.rhs[tid] : 0.0;
  if (tid == 0) flag = 0;
  __syncthreads();
  if (!factor_block(sm, &flag, L.Linv, L.rhs, kb, tid) && tid == 0) St->chol_ok = 0;
}

// Step k of the right-looking factorization, one workgroup per block (i, j), k < j <= i, of what is left. Block k's
// inverse X is known, so each workgroup forms the panel blocks it needs itself, L_ik = A_ik X^T and L_jk = A_jk X^T, and
// subtracts L_ik L_jk^T from A_ij: recomputing a panel block costs a 64-wide product (10 of 16 tiles, X being
// triangular), less than the launch that a separate panel kernel would cost. The workgroup of (i, i) also keeps L_ik,
// transposed, in the unused upper triangle (block (k, i); the lower A_ik is still read by others) for the backward
// solve, and takes e_i -= L_ik y_k. The first workgroup, block (k + 1, k + 1), goes on to factor its block
// (factor_block), so the next step starts with its inverse: one launch per block column, bound by that workgroup's serial
// chain. Order 1194: 23 us per block column, against 45 us with separate diagonal, panel and trailing launches (24 + 11
// + 10); order 336: 22 against 43. In a large system the trailing updates take over, where the recomputed panels cost
// what the launches save: gather, factor and backward solve per iteration, here against separate launches, order 2394
// 1.38 against 2.36 ms, 3594 2.85 against 4.20, 4794 5.16 against 6.64, 6114 (1020 key frames, the most a window may hold
// is 1024) 10.1 against 10.3. So one rule serves every order.
__global__ __launch_bounds__(256) void k_lstep(Batch b, int w, int k) {
  __shared__ double sm[3 * 16 * kTs];
  __shared__ double sy[kLB], sred[4 * kLB];
  __shared__ int flag;
  static_assert(kFbWords <= 3 * 16 * kTs, "factor_block reuses the staging memory");
  const WindowDesc W = b.win[w];
  WindowState* St = b.st + w;
  if (St->done || !St->chol_ok) return;
  const Large L = large_of(b, W);
  const int n = L.n, k0 = kLB * k, tid = threadIdx.x;  // block k is a full one: blocks follow it
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int at = kTr * (lane >> 4) + (lane & 15);
  int ii = 0, jj = blockIdx.x;  // 0 <= jj <= ii, row by row
  while (jj > ii) jj -= ++ii;
  const bool diag = ii == jj;
  const int i0 = kLB * (k + 1 + ii), j0 = kLB * (k + 1 + jj);
  const int ib = min(kLB, n - i0), jb = min(kLB, n - j0);
  double* sX = sm;                // X
  double* sA = sm + 16 * kTs;     // A_ik, then L_ik
  double* sB = diag ? sA : sm + 32 * kTs;  // A_jk, then L_jk
  if (tid == 0) flag = 0;
  stage_transposed(sX, L.Linv + static_cast<int64_t>(k) * kLB * kLB, kLB, kLB, kLB, tid);
  stage_transposed(sA, L.A + static_cast<int64_t>(i0) * n + k0, n, ib, kLB, tid);
  if (!diag) stage_transposed(sB, L.A + static_cast<int64_t>(j0) * n + k0, n, jb, kLB, tid);
  if (tid < kLB) sy[tid] = L.rhs[k0 + tid];
  // this wavefront's tiles (wave, J) of A_ij, element (4 v + lane / 16, lane % 16) in register v
  double4v acc[4];
#pragma unroll
  for (int J = 0; J < 4; ++J)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      // a diagonal block: symmetric, read from its lower triangle, identity past the matrix
      const int r0 = 16 * wave + 4 * v + (lane >> 4), c0 = 16 * J + (lane & 15);
      const int r = diag ? max(r0, c0) : r0, c = diag ? min(r0, c0) : c0;
      acc[J][v] = (r0 < ib && c0 < jb) ? L.A[static_cast<int64_t>(i0 + r) * n + j0 + c] : (diag && r0 == c0 ? 1.0 : 0.0);
    }
  __syncthreads();
  // The transposed panel tiles (L_ik^T)(J, wave) = sum_M X(J, M) A_ik(wave, M)^T come out in the staged layout; they
  // replace the tiles (wave, J) of A_ik, which only this wavefront reads.
  auto panel = [&](double* sS) {
    double4v p[4];
#pragma unroll
    for (int J = 0; J < 4; ++J) {
      p[J] = double4v{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int M = 0; M <= J; ++M)
        p[J] = staged_update(p[J], sX + kTs * (4 * J + M), sS + kTs * (4 * wave + M), at);
    }
    wave_lds_sync();
#pragma unroll
    for (int J = 0; J < 4; ++J)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        p[J][v] = -p[J][v];
        sS[kTs * (4 * wave + J) + 4 * kTr * v + at] = p[J][v];
      }
    return [=](int J, int v) { return p[J][v]; };
  };
  const auto pi = panel(sA);
  if (!diag) {
    panel(sB);
  } else {
#pragma unroll
    for (int J = 0; J < 4; ++J)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int c = 16 * J + 4 * v + (lane >> 4), r = 16 * wave + (lane & 15);
        if (r < ib) L.A[static_cast<int64_t>(k0 + c) * n + i0 + r] = pi(J, v);
      }
  }
  __syncthreads();
#pragma unroll
  for (int J = 0; J < 4; ++J)
#pragma unroll
    for (int M = 0; M < 4; ++M)
      acc[J] = staged_update(acc[J], sA + kTs * (4 * wave + M), sB + kTs * (4 * J + M), at);
  double e = 0.0;
  if (diag) {  // e_i -= L_ik y_k: wavefront g sums columns 16 g .. 16 g + 15 of row `lane`
    double s = 0.0;
#pragma unroll
    for (int m = 0; m < 16; ++m) s += sA[kTs * (4 * (lane >> 4) + wave) + kTr * m + (lane & 15)] * sy[16 * wave + m];
    sred[kLB * wave + lane] = s;
    __syncthreads();
    if (tid < ib) e = L.rhs[i0 + tid] - ((sred[tid] + sred[kLB + tid]) + (sred[2 * kLB + tid] + sred[3 * kLB + tid]));
  }
  if (blockIdx.x != 0) {
#pragma unroll
    for (int J = 0; J < 4; ++J)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = 16 * wave + 4 * v + (lane >> 4), c = 16 * J + (lane & 15);
        if (r < ib && c < jb && (!diag || c <= r)) L.A[static_cast<int64_t>(i0 + r) * n + j0 + c] = acc[J][v];
      }
    if (diag && tid < ib) L.rhs[i0 + tid] = e;
    return;
  }
  // block (k + 1, k + 1): its upper tiles and right-hand side to factor_block (the barrier above ended the reads of sm)
#pragma unroll
  for (int J = 0; J < 4; ++J) {
    if (J < wave) continue;
    double* dst = J == wave ? sm + kFbDg + 256 * J : sm + kFbU + 256 * pair_of(wave, J);
#pragma unroll
    for (int v = 0; v < 4; ++v) dst[64 * v + lane] = acc[J][v];
  }
  if (tid < kLB) sm[kFbVec + tid] = e;
  __syncthreads();
  if (!factor_block(sm, &flag, L.Linv + static_cast<int64_t>(k + 1) * kLB * kLB, L.rhs + i0, ib, tid) && tid == 0)
    St->chol_ok = 0;
}

// Backward substitution L^T x = y in one workgroup of 1024 threads, 64-row blocks from the last, then the pose step, its
// max-norm, dc^T diag(U) dc and the trial key frames. For block bk, r = y_bk - sum_{i past the block} L[i][block bk]^T
// x_i: the rows of L^T lie in the upper triangle (k_lstep), so each of the 16 wavefronts takes four rows with its lanes
// along them, 16 loads of 16 bytes of a lane in flight, and adds its lanes; then x_bk = X_bk^T r with the kept
// inverse, whose loads do not wait for r. x stays in the dynamic shared memory (n doubles). The latency of one
// workgroup's loads bounds it: order 1194, 5.7 MB, 101 us, the epilogue (8 us as a launch of its own) included; 110 us
// with the rows gathered down the columns of L, 141 with 8-byte loads along the rows.
__global__ __launch_bounds__(1024) void k_bsolve(Batch b, int w) {
  constexpr int kG = 16;             // wavefronts
  constexpr int kR = kLB / kG;       // rows of a block per wavefront
  extern __shared__ double sx[];     // y, overwritten by x block by block
  __shared__ double part[kG * kLB];
  __shared__ double sr[kLB];
  __shared__ double red[2 * kG];
  const WindowDesc W = b.win[w];
  WindowState* St = b.st + w;
  if (St->done || !St->chol_ok) return;
  const Large L = large_of(b, W);
  const int n = L.n, tid = threadIdx.x, c = tid & 63, g = tid >> 6;
  const int nb = (n + kLB - 1) / kLB;
  for (int i = tid; i < n; i += blockDim.x) sx[i] = L.rhs[i];
  __syncthreads();
  for (int bk = nb - 1; bk >= 0; --bk) {
    const int b0 = kLB * bk, bb = min(kLB, n - b0);
    // rows kR g .. kR g + kR - 1 of X_bk (zero above the diagonal), column c
    const double* X = L.Linv + static_cast<int64_t>(bk) * kLB * kLB + kR * g * kLB + c;
    double xv[kR];
#pragma unroll
    for (int r = 0; r < kR; ++r) xv[r] = X[r * kLB];
    double s[kR] = {};
    // rows past the matrix (only in the last block, which has nothing past it) are not reached
    const double2* row = reinterpret_cast<const double2*>(L.A + static_cast<int64_t>(b0 + kR * g) * n);
    const int h = n / 2;  // n is even (6 per key frame), so rows and column pairs are 16-byte aligned
    for (int i = (b0 + kLB) / 2 + c; i < h; i += 4 * 64) {
      double2 v[4][kR];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int r = 0; r < kR; ++r) v[u][r] = row[static_cast<int64_t>(r) * h + min(i + 64 * u, h - 1)];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int q = i + 64 * u;
        const double x0 = q < h ? sx[2 * q] : 0.0, x1 = q < h ? sx[2 * q + 1] : 0.0;
#pragma unroll
        for (int r = 0; r < kR; ++r) s[r] += v[u][r].x * x0 + v[u][r].y * x1;
      }
    }
    // the four rows' sums over the lanes: lanes exchange two rows, then one, so that each 16 lanes end with one row
    static_assert(kR == 4, "the exchange below covers four rows");
    const bool hi = c & 32, odd = c & 16;
    const double t0 = hi ? s[2] : s[0], t1 = hi ? s[3] : s[1];
    const double q0 = t0 + __shfl_xor(hi ? s[0] : s[2], 32), q1 = t1 + __shfl_xor(hi ? s[1] : s[3], 32);
    const double sum = sum_row16_dpp((odd ? q1 : q0) + __shfl_xor(odd ? q0 : q1, 16));
    if ((c & 15) == 0) {
      const int r = kR * g + (c >> 4);
      sr[r] = r < bb ? sx[b0 + r] - sum : 0.0;
    }
    __syncthreads();
    // x_c = sum_{m >= c} X[m][c] r_m, four rows per wavefront, added in wavefront order
    double xs = 0.0;
#pragma unroll
    for (int r = 0; r < kR; ++r) xs += xv[r] * sr[kR * g + r];
    part[g * kLB + c] = xs;
    __syncthreads();
    if (tid < bb) {
      double x = 0.0;
#pragma unroll
      for (int q = 0; q < kG; ++q) x += part[q * kLB + c];
      sx[b0 + c] = x;
    }
    __syncthreads();
  }
  double sc = 0.0;
  float mx = 0.f;
  for (int i = tid; i < n; i += blockDim.x) {
    const double x = sx[i];
    b.dc[W.dc_off + i] = static_cast<float>(x);
    b.dc64[W.dc_off + i] = x;
    sc += x * x * L.du[i];
    mx = fmaxf(mx, fabsf(static_cast<float>(x)));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    sc += __shfl_xor(sc, o);
    mx = fmaxf(mx, __shfl_xor(mx, o));
  }
  if (c == 0) {
    red[g] = sc;
    red[kG + g] = static_cast<double>(mx);
  }
  __syncthreads();
  if (tid == 0) {
    double t = 0.0, m = 0.0;
    for (int q = 0; q < kG; ++q) {
      t += red[q];
      m = fmax(m, red[kG + q]);
    }
    St->scal_pose = t;
    St->maxdc = static_cast<float>(m);
  }
  write_trial_poses(b, W, St->cur, sx, tid, blockDim.x);
}

namespace sba_dev {

// The factor and solve of window w (n = 6 free key frames): gather, blocked Cholesky, backward solve and epilogue. One
// launch per 64-row block and two besides.
hipError_t launch_large_factor(const Batch& b, int w, int n, hipStream_t s) {
  const int nb = (n + kLB - 1) / kLB, ncf = n / 6;
  hipLaunchKernelGGL(k_gather, dim3(ncf * (ncf + 1) / 2), dim3(64 * kGatherWaves), 0, s, b, w);
  hipLaunchKernelGGL(k_lfirst, dim3(1), dim3(256), 0, s, b, w);
  hipError_t e = hipGetLastError();
  for (int k = 0; k + 1 < nb && e == hipSuccess; ++k) {
    const int m = nb - k - 1;
    hipLaunchKernelGGL(k_lstep, dim3(m * (m + 1) / 2), dim3(256), 0, s, b, w, k);
    e = hipGetLastError();
  }
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_bsolve, dim3(1), dim3(1024), sizeof(double) * n, s, b, w);
  return hipGetLastError();
}

}  // namespace sba_dev
