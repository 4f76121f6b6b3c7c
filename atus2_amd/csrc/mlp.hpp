// mlp.hpp -- launchers of the warm-start network kernels (k_mlp.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace atus {

// what a product's tiles do with their sums
struct GemmEpilogue {
  const float* bias = nullptr;  // added per column
  int act = 0;                  // 1: tanh; 2: times (1 - X^2), X laid out as C
  const float* X = nullptr;
  // loss layer: d = sum + bias - T[idx[m]][n] (idx NULL: T[m]), C = scale d,
  // loss[tile] = sum of d^2 over the tile (mlp_loss_parts of them)
  const float* T = nullptr;
  const int* idx = nullptr;
  float scale = 0.f;
  float* loss = nullptr;
  float* colsum = nullptr;      // column sums of B
};
constexpr int MLP_TILE = 64;   // rows and columns of a product's tile
constexpr int MLP_SLICE = 32;  // its slices along k
// floats of workspace mlp_gemm needs for an M x N x K product, with or without
// column sums
size_t mlp_gemm_work(int M, int N, int K, bool colsum = false);
// loss partials of an M x N output
size_t mlp_loss_parts(int M, int N);
// C (M x N, row-major) from A B; A(m,k) = A[m*sam + k*sak], B(k,n) =
// B[k*sbk + n*sbn]; operands rounded to bf16 (split: hi + lo bf16 pairs,
// three products), fp32 accumulation
hipError_t mlp_gemm(const float* A, long long sam, long long sak, const float* B, long long sbk, long long sbn,
                    float* C, int M, int N, int K, const GemmEpilogue& e, float* work, size_t work_floats,
                    hipStream_t s, bool split);
// loss[slot] = sum of part[0..nb) / n; not finite: *bad = 1
hipError_t mlp_loss(const float* part, int nb, double n, float* loss, int slot, int* bad, hipStream_t s);
// does nothing once *bad is set
hipError_t mlp_adam(float* p, const float* g, float* m, float* v, long long n, float lr, float b1, float b2,
                    float eps, float c1, float c2, const int* bad, hipStream_t s);
hipError_t mlp_gather(const float* src, const int* idx, int rows, long long w, float* dst, hipStream_t s);
// psi[n0][n1][n2] = sum E0[i0][j0] E1[i1][j1] E2[i2][j2] y[j0][j1][j2] over the
// 32^3 values y, through t1 (n0 x 32 x 32) and t2 (n0 x n1 x 32); E_a: n_a x 32
hipError_t mlp_interp32(const float* y, const double* E0, const double* E1, const double* E2, double* t1, double* t2,
                        double2* psi, const int n[3], hipStream_t s);

}  // namespace atus
