// The 16 x 16 tile factor of the FP64 kernels (sba_tiles.h) on tiles whose second and fourth rows of every panel cancel
// to a given part of their diagonal entry: A = U^T U and X = U^-T in extended precision against the bounds of Cholesky
// and of substitution, which do not grow with the condition of the tile, and no infinities in a factor reported good.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <limits>
#include <random>
#include <vector>

#include "../../cuvslam_amd/csrc/sba_tiles.h"

__global__ __launch_bounds__(64) void factor(const double* A, double* U, double* X, double* rdiag, int* ok) {
  __shared__ double xt[256];
  const int lane = threadIdx.x;
  const size_t at = 256 * static_cast<size_t>(blockIdx.x);
  sba_tiles::double4v t;
  for (int v = 0; v < 4; ++v) t[v] = A[at + 64 * v + lane];
  const bool good = sba_tiles::factor_tile(t, xt, rdiag + 16 * blockIdx.x, lane);
  sba_tiles::wave_lds_sync();
  for (int v = 0; v < 4; ++v) {
    U[at + 64 * v + lane] = t[v];
    X[at + 64 * v + lane] = xt[64 * v + lane];  // X^T, row-major
  }
  if (lane == 0) ok[blockIdx.x] = good;
}

int main() {
  constexpr int kTiles = 500;
  const double eps = std::numeric_limits<double>::epsilon() / 2;
  // Higham, Accuracy and Stability, theorems 10.3 (|U^T U - A| <= c |U^T| |U|, so c sqrt(a_ii a_jj)) and 8.5
  // (|U^T X - I| <= c |U^T| |X|), c = (16 + 1) eps; doubled, since a quotient is a product with a rounded reciprocal
  const double bound = 2 * 17 * eps;
  std::vector<double> A(256 * kTiles), U(A.size()), X(A.size()), r(16 * kTiles);
  std::vector<int> ok(kTiles);
  double *dA, *dU, *dX, *dr;
  int* dok;
  const size_t bytes = A.size() * sizeof(double);
  if (hipMalloc(&dA, bytes) || hipMalloc(&dU, bytes) || hipMalloc(&dX, bytes) || hipMalloc(&dr, r.size() * sizeof(double)) ||
      hipMalloc(&dok, ok.size() * sizeof(int)))
    return 2;
  int failures = 0;
  for (int pos : {-1, 1, 3})  // row of the panel that cancels; -1: none
    for (double part : {1.0, 1e-4, 1e-8, 1e-12, 1e-15}) {
      if ((pos < 0) != (part == 1.0)) continue;
      std::mt19937_64 g(11);
      std::normal_distribution<double> normal;
      for (int m = 0; m < kTiles; ++m) {
        double L[16][16] = {};
        for (int i = 0; i < 16; ++i) {
          double s = 0;
          for (int j = 0; j < i; ++j) {
            L[i][j] = normal(g);
            s += L[i][j] * L[i][j];
          }
          L[i][i] = (i & 3) == pos ? std::sqrt(part * std::max(s, 1.0)) : 1 + std::fabs(normal(g));
        }
        for (int i = 0; i < 16; ++i)
          for (int j = 0; j <= i; ++j) {
            long double a = 0;
            for (int k = 0; k < 16; ++k) a += static_cast<long double>(L[i][k]) * L[j][k];
            A[256 * m + 16 * i + j] = A[256 * m + 16 * j + i] = static_cast<double>(a);
          }
      }
      if (hipMemcpy(dA, A.data(), bytes, hipMemcpyHostToDevice)) return 2;
      hipLaunchKernelGGL(factor, dim3(kTiles), dim3(64), 0, 0, dA, dU, dX, dr, dok);
      if (hipGetLastError() || hipMemcpy(U.data(), dU, bytes, hipMemcpyDeviceToHost) ||
          hipMemcpy(X.data(), dX, bytes, hipMemcpyDeviceToHost) ||
          hipMemcpy(r.data(), dr, r.size() * sizeof(double), hipMemcpyDeviceToHost) ||
          hipMemcpy(ok.data(), dok, ok.size() * sizeof(int), hipMemcpyDeviceToHost))
        return 2;
      int good = 0;
      double eu = 0, ex = 0, er = 0;  // NaN counts as a failure of the comparisons below
      for (int m = 0; m < kTiles; ++m) {
        if (!ok[m]) continue;
        ++good;
        const double *u = &U[256 * m], *x = &X[256 * m], *a = &A[256 * m];
        auto worse = [](double& worst, double e) { worst = e <= worst ? worst : e; };
        for (int i = 0; i < 16; ++i) {
          worse(er, std::fabs(r[16 * m + i] * u[17 * i] - 1));
          for (int j = 0; j < 16; ++j) {
            long double uu = 0, ux = 0, mag = 0;
            for (int k = 0; k < 16; ++k) {
              uu += static_cast<long double>(u[16 * k + i]) * u[16 * k + j];
              const long double p = static_cast<long double>(u[16 * k + i]) * x[16 * j + k];
              ux += p;
              mag += std::fabs(p);
            }
            worse(eu, static_cast<double>(std::fabs(uu - a[16 * i + j]) / std::sqrt(a[17 * i] * a[17 * j])));
            // no error is possible where every product is an exact zero
            const long double d = std::fabs(ux - (i == j));
            worse(ex, d == 0 ? 0 : static_cast<double>(d / mag));
          }
        }
      }
      // tiles that stay positive definite in rounded arithmetic: all of them down to 1e-4, but for a few
      const bool pass = eu <= bound && ex <= bound && er <= bound && good >= (part >= 1e-4 ? kTiles - 10 : 1);
      failures += !pass;
      std::printf("row %2d, part %.0e: %d good, |U^T U - A| %.1e, |U^T X - I| %.1e, 1 / U_ii %.1e: %s\n", pos, part, good, eu,
                  ex, er, pass ? "ok" : "FAILED");
    }
  std::printf("%s (bound %.1e)\n", failures ? "FAILED" : "OK", bound);
  return failures != 0;
}
