// k_mlp.hip -- kernels of the warm-start network: BF16 MFMA matrix
// products with FP32 accumulation (v_mfma_f32_16x16x32_bf16), their
// epilogues, the loss, the optimiser, and the separable interpolation of
// the network's 32^3 output onto a solver grid.
#include "launch.hpp"
#include "mlp.hpp"

namespace atus {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- products
// C(m,n) = sum_k A(m,k) B(k,n), A(m,k) = A[m*sam + k*sak], B(k,n) =
// B[k*sbk + n*sbn], operands rounded to bf16 (SPLIT false) or split as a = hi
// + lo, hi = bf16(a), lo = bf16(a - hi), with a b ~ hi_a hi_b + hi_a lo_b +
// lo_a hi_b (SPLIT true: three products, about 16 significant bits per
// operand), fp32 accumulation.
//
// A workgroup of four wavefronts forms a 64 x 64 tile in slices of 32 along
// k.  An operand's slice goes through LDS as [row][k], 8 consecutive k of a
// row per 16-byte write, so each element is read from memory and split once
// per tile instead of once per 16 x 16 tile and wavefront; the next slice is
// in flight in registers while this one is multiplied.  The large products
// (256 x 32768 x 64 and its two transposes) stream their operands; what
// follows them rides in their epilogues rather than in passes of its own.
constexpr int GT = MLP_TILE;  // tile edge
constexpr int GK = MLP_SLICE; // slice along k
constexpr int GP = GK + 8;    // LDS row pitch: 16-byte rows on distinct banks

enum GemmMode {
  G_OUT = 0,    // C = act(sum + bias)
  G_PART = 1,   // P[blockIdx.z][m][n]: partial sums of a split along k; the
                // column sums' partials [blockIdx.z][n] behind them
  G_MSE = 2     // d = sum + bias - T[row(m)][n]: C = 2 d / count, loss partials
};

struct GemmArgs {
  const float* A;
  long long sam, sak;
  const float* B;
  long long sbk, sbn;
  float* C;
  int M, N, K, kchunk;
  int mode;
  GemmEpilogue e;
};

// 8 values of an operand's row r at k0..k0+7 (0 beyond the matrix)
__device__ __forceinline__ void gemm_load(float (&f)[8], const float* src, long long sr, long long sk, int r, int rows,
                                          int k0, int ke, bool vec) {
  const float* p = src + (long long)r * sr + (long long)k0 * sk;
  if (vec && r < rows && k0 + 8 <= ke) {
    const float4 x = *reinterpret_cast<const float4*>(p), y = *reinterpret_cast<const float4*>(p + 4);
    f[0] = x.x, f[1] = x.y, f[2] = x.z, f[3] = x.w;
    f[4] = y.x, f[5] = y.y, f[6] = y.z, f[7] = y.w;
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] = (r < rows && k0 + j < ke) ? p[(long long)j * sk] : 0.f;
  }
}

template <bool SPLIT>
__device__ __forceinline__ void gemm_store(const float (&f)[8], __bf16* hi, __bf16* lo, int at) {
  bf16x8 h, l;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    h[j] = (__bf16)f[j];
    if constexpr (SPLIT) l[j] = (__bf16)(f[j] - (float)h[j]);
  }
  *reinterpret_cast<bf16x8*>(hi + at) = h;
  if constexpr (SPLIT) *reinterpret_cast<bf16x8*>(lo + at) = l;
}

__device__ __forceinline__ float gemm_act(float s, int act, const float* X, long long at) {
  if (act == 1) return tanhf(s);
  if (act == 2) return s * (1.f - X[at] * X[at]);  // dZ = dX (1 - X^2), X = tanh(Z)
  return s;
}

template <bool SPLIT>
__global__ __launch_bounds__(256) void k_gemm_bf16(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) __bf16 sh[SPLIT ? 4 : 2][GT * GP];
  __shared__ float red[256];
  __bf16* ah = sh[0];
  __bf16* bh = sh[1];
  __bf16* al = sh[SPLIT ? 2 : 0];
  __bf16* bl = sh[SPLIT ? 3 : 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n0 = blockIdx.x * GT, m0 = blockIdx.y * GT;
  const int kb = blockIdx.z * g.kchunk, ke = min(g.K, kb + g.kchunk);
  // this thread's share of a slice: 8 k of one row of each operand.  Rows
  // run over the lanes where the operand is contiguous along them, k
  // groups where it is contiguous along k.
  const bool ak = g.sak == 1, bk = g.sbk == 1;
  const int ar = ak ? tid >> 2 : tid & 63, ag = ak ? tid & 3 : tid >> 6;
  const int br = bk ? tid >> 2 : tid & 63, bg = bk ? tid & 3 : tid >> 6;
  const bool av = ak && (g.sam & 3) == 0 && ((unsigned long long)g.A & 15) == 0;
  const bool bv = bk && (g.sbn & 3) == 0 && ((unsigned long long)g.B & 15) == 0;
  float fa[8], fb[8], bsum = 0.f;
  f32x4 acc[2][2] = {};
  const int i = lane & 15, grp = lane >> 4;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  gemm_load(fa, g.A, g.sam, g.sak, m0 + ar, g.M, kb + 8 * ag, ke, av);
  gemm_load(fb, g.B, g.sbn, g.sbk, n0 + br, g.N, kb + 8 * bg, ke, bv);
  for (int k0 = kb; k0 < ke; k0 += GK) {
    __syncthreads();  // the last slice's reads are done
    gemm_store<SPLIT>(fa, ah, al, ar * GP + 8 * ag);
    gemm_store<SPLIT>(fb, bh, bl, br * GP + 8 * bg);
#pragma unroll
    for (int j = 0; j < 8; ++j) bsum += fb[j];
    __syncthreads();
    if (k0 + GK < ke) {
      gemm_load(fa, g.A, g.sam, g.sak, m0 + ar, g.M, k0 + GK + 8 * ag, ke, av);
      gemm_load(fb, g.B, g.sbn, g.sbk, n0 + br, g.N, k0 + GK + 8 * bg, ke, bv);
    }
    bf16x8 a[2], b[2], a2[2], b2[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int oa = (wm + 16 * t + i) * GP + 8 * grp, ob = (wn + 16 * t + i) * GP + 8 * grp;
      a[t] = *reinterpret_cast<const bf16x8*>(ah + oa);
      b[t] = *reinterpret_cast<const bf16x8*>(bh + ob);
      if constexpr (SPLIT) {
        a2[t] = *reinterpret_cast<const bf16x8*>(al + oa);
        b2[t] = *reinterpret_cast<const bf16x8*>(bl + ob);
      }
    }
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y) {
        if constexpr (SPLIT) {
          acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2[x], b[y], acc[x][y], 0, 0, 0);
          acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[x], b2[y], acc[x][y], 0, 0, 0);
        }
        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[x], b[y], acc[x][y], 0, 0, 0);
      }
  }
  // lane l holds rows 4 (l/16) + 0..3 of column l%16 of each 16 x 16 tile
  float loss = 0.f;
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm + 16 * x + 4 * grp + r, col = n0 + wn + 16 * y + i;
        if (row >= g.M || col >= g.N) continue;
        const long long at = (long long)row * g.N + col;
        if (g.mode == G_PART) {
          g.C[(long long)blockIdx.z * g.M * g.N + at] = acc[x][y][r];
        } else {
          float s = acc[x][y][r];
          if (g.e.bias) s += g.e.bias[col];
          if (g.mode == G_MSE) {
            const float d = s - g.e.T[(long long)(g.e.idx ? g.e.idx[row] : row) * g.N + col];
            g.C[at] = g.e.scale * d;
            loss += d * d;
          } else {
            g.C[at] = gemm_act(s, g.e.act, g.e.X, at);
          }
        }
      }
  if (g.mode == G_MSE) {
    red[tid] = loss;
    __syncthreads();
    for (int q = 128; q > 0; q >>= 1) {
      if (tid < q) red[tid] += red[tid + q];
      __syncthreads();
    }
    if (tid == 0) g.e.loss[blockIdx.y * gridDim.x + blockIdx.x] = red[0];
  }
  if (g.e.colsum && blockIdx.y == 0) {
    // column sums of B (one slice group per wavefront or lane quad)
    red[tid] = bsum;
    __syncthreads();
    if (tid < GT && n0 + tid < g.N) {
      float s = 0.f;
#pragma unroll
      for (int q = 0; q < 4; ++q) s += red[bk ? 4 * tid + q : tid + GT * q];
      float* o = g.mode == G_PART ? g.C + (long long)gridDim.z * g.M * g.N + (long long)blockIdx.z * g.N : g.e.colsum;
      o[n0 + tid] = s;
    }
  }
}

// C[m][n] = act(sum_z P[z][m][n] + bias[n]), and the column sums from their
// partials: 64 elements per workgroup, each wavefront a quarter of the
// splits, 8 loads in flight, in a fixed order (64 splits of 256 x 64 one
// after another in a thread took 16 us)
__global__ __launch_bounds__(256) void k_gemm_sum(const float* __restrict__ P, int splits, int M, int N,
                                                  GemmEpilogue ep, float* __restrict__ C) {
  __shared__ float sh[4][64];
  const long long MN = (long long)M * N, all = MN + (ep.colsum ? N : 0);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int per = (splits + 3) / 4, z0 = w * per, z1 = min(splits, z0 + per);
  for (long long e0 = (long long)blockIdx.x * 64; e0 < all; e0 += (long long)gridDim.x * 64) {
    const long long e = e0 + l;
    const long long step = e < MN ? MN : N;
    const float* p = e < MN ? P + e : P + splits * MN + (e - MN);
    float s = 0.f;
    if (e < all) {
      int z = z0;
      for (; z + 8 <= z1; z += 8) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = p[(z + i) * step];
#pragma unroll
        for (int i = 0; i < 8; ++i) s += v[i];
      }
      for (; z < z1; ++z) s += p[z * step];
    }
    sh[w][l] = s;
    __syncthreads();
    if (w == 0 && e < all) {
      s = (sh[0][l] + sh[1][l]) + (sh[2][l] + sh[3][l]);
      if (e >= MN) {
        ep.colsum[e - MN] = s;
      } else {
        if (ep.bias) s += ep.bias[e % N];
        C[e] = gemm_act(s, ep.act, ep.X, e);
      }
    }
    __syncthreads();
  }
}

// mean squared error of step `slot`: loss[slot] = sum of the nb partials / n
// (fixed order); a value that is not finite sets *bad, which stays set and
// keeps Adam from changing the parameters from then on
__global__ __launch_bounds__(256) void k_loss(const float* __restrict__ part, int nb, double n, float* __restrict__ loss,
                                              int slot, int* __restrict__ bad) {
  __shared__ double sh[256];
  double acc = 0.0;
  for (int b = threadIdx.x; b < nb; b += 256) acc += part[b];
  sh[threadIdx.x] = acc;
  __syncthreads();
  for (int q = 128; q > 0; q >>= 1) {
    if ((int)threadIdx.x < q) sh[threadIdx.x] += sh[threadIdx.x + q];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double l = sh[0] / n;
    loss[slot] = (float)l;
    if (!isfinite(l)) *bad = 1;
  }
}

// Adam (Kingma & Ba 2015) with bias corrections c1 = 1 - beta1^t, c2 = 1 - beta2^t
__global__ __launch_bounds__(256) void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                                              float* __restrict__ v, long long n, float lr, float b1, float b2,
                                              float eps, float c1, float c2, const int* __restrict__ bad) {
  if (*bad) return;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long long)gridDim.x * blockDim.x) {
    const float ge = g[e];
    const float me = b1 * m[e] + (1.f - b1) * ge;
    const float ve = b2 * v[e] + (1.f - b2) * ge * ge;
    m[e] = me;
    v[e] = ve;
    p[e] -= lr * (me / c1) / (sqrtf(ve / c2) + eps);
  }
}

// rows idx[r] of src (n x w) into dst (rows x w)
__global__ __launch_bounds__(256) void k_gather(const float* __restrict__ src, const int* __restrict__ idx, int rows,
                                                long long w, float* __restrict__ dst) {
  const long long tot = (long long)rows * w;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < tot; e += (long long)gridDim.x * blockDim.x)
    dst[e] = src[(long long)idx[e / w] * w + e % w];
}

// one axis of a separable interpolation: out[p][i][q] = sum_j E[i][j] in[p][j][q]
// (p < outer, i < nout, j < nin, q < inner); `in` is fp32 (the network's
// output) or fp64, out is fp64 or, for the last axis, the complex field
template <typename Tin, bool TO_FIELD>
__global__ __launch_bounds__(256) void k_interp_axis(const Tin* __restrict__ in, const double* __restrict__ E,
                                                     void* __restrict__ out, long long outer, int nin, int nout,
                                                     long long inner) {
  const long long tot = outer * nout * inner;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < tot; e += (long long)gridDim.x * blockDim.x) {
    const long long q = e % inner;
    const long long r = e / inner;
    const int i = (int)(r % nout);
    const long long p = r / nout;
    const double* Ei = E + (long long)i * nin;
    const Tin* src = in + p * nin * inner + q;
    double acc = 0.0;
    for (int j = 0; j < nin; ++j) acc += Ei[j] * (double)src[(long long)j * inner];
    if constexpr (TO_FIELD)
      static_cast<double2*>(out)[e] = make_double2(acc, 0.0);
    else
      static_cast<double*>(out)[e] = acc;
  }
}

}  // namespace atus

namespace atus {

static unsigned ew_grid(long long n) {
  long long b = (n + 255) / 256;
  if (b > 8192) b = 8192;
  if (b < 1) b = 1;
  return (unsigned)b;
}

// Split of K: products of fewer tiles than CUs and more than 8 slices give
// every CU a tile of at least 8 slices of its own (256 x 64 x 32768: 64
// splits of 16 slices, 256 workgroups); shorter ones are not worth the second
// launch.  Weight gradients of large batches split too: unsplit, 65536 rows
// were a chain of 2048 slices in as few workgroups as the layer has tiles
// (4-256-256-64-256: 10.1 ms per step, 0.88 split)
static void split_plan(int M, int N, int K, int* splits, int* kchunk) {
  const long long tiles = (long long)((M + GT - 1) / GT) * ((N + GT - 1) / GT);
  const int slices = (K + GK - 1) / GK;
  long long want = tiles < CU_COUNT ? (CU_COUNT + tiles - 1) / tiles : 1;
  if (want > slices / 8) want = slices / 8;
  if (want < 1) want = 1;
  const int per = (int)((slices + want - 1) / want);
  *kchunk = per * GK;
  *splits = (slices + per - 1) / per;
}

size_t mlp_gemm_work(int M, int N, int K, bool colsum) {
  int splits, kchunk;
  split_plan(M, N, K, &splits, &kchunk);
  return splits > 1 ? (size_t)splits * (M + (colsum ? 1 : 0)) * N : 0;
}

size_t mlp_loss_parts(int M, int N) { return (size_t)((M + GT - 1) / GT) * ((N + GT - 1) / GT); }

hipError_t mlp_gemm(const float* A, long long sam, long long sak, const float* B, long long sbk, long long sbn,
                    float* C, int M, int N, int K, const GemmEpilogue& e, float* work, size_t work_floats,
                    hipStream_t s, bool split) {
  if (M < 1 || N < 1 || K < 1) return hipErrorInvalidValue;
  int splits, kchunk;
  split_plan(M, N, K, &splits, &kchunk);
  if (e.T) {
    // the loss needs the whole of K in one workgroup
    splits = 1;
    kchunk = K;
  }
  if (splits > 1 && mlp_gemm_work(M, N, K, e.colsum != nullptr) > work_floats) return hipErrorInvalidValue;
  GemmArgs g{A, sam, sak, B, sbk, sbn, splits > 1 ? work : C, M, N, K, kchunk, splits > 1 ? G_PART : e.T ? G_MSE : G_OUT,
             e};
  const long long tm = (M + GT - 1) / GT, tn = (N + GT - 1) / GT;
  if (tm > 65535) return hipErrorInvalidValue;
  const dim3 grid((unsigned)tn, (unsigned)tm, (unsigned)splits);
  if (split)
    hipLaunchKernelGGL(k_gemm_bf16<true>, grid, dim3(256), 0, s, g);
  else
    hipLaunchKernelGGL(k_gemm_bf16<false>, grid, dim3(256), 0, s, g);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess || splits == 1) return err;
  hipLaunchKernelGGL(k_gemm_sum, dim3(ew_grid(((long long)M + (e.colsum ? 1 : 0)) * N * 4)), dim3(256), 0, s, work, splits,
                     M, N, e, C);
  return hipGetLastError();
}

hipError_t mlp_loss(const float* part, int nb, double n, float* loss, int slot, int* bad, hipStream_t s) {
  hipLaunchKernelGGL(k_loss, dim3(1), dim3(256), 0, s, part, nb, n, loss, slot, bad);
  return hipGetLastError();
}

hipError_t mlp_adam(float* p, const float* g, float* m, float* v, long long n, float lr, float b1, float b2,
                    float eps, float c1, float c2, const int* bad, hipStream_t s) {
  hipLaunchKernelGGL(k_adam, dim3(ew_grid(n)), dim3(256), 0, s, p, g, m, v, n, lr, b1, b2, eps, c1, c2, bad);
  return hipGetLastError();
}

hipError_t mlp_gather(const float* src, const int* idx, int rows, long long w, float* dst, hipStream_t s) {
  hipLaunchKernelGGL(k_gather, dim3(ew_grid((long long)rows * w)), dim3(256), 0, s, src, idx, rows, w, dst);
  return hipGetLastError();
}

hipError_t mlp_interp32(const float* y, const double* E0, const double* E1, const double* E2, double* t1, double* t2,
                        double2* psi, const int n[3], hipStream_t s) {
  // [32][32][32] -> [n0][32][32] -> [n0][n1][32] -> [n0][n1][n2]
  hipLaunchKernelGGL((k_interp_axis<float, false>), dim3(ew_grid((long long)n[0] * 32 * 32)), dim3(256), 0, s, y, E0,
                     (void*)t1, 1LL, 32, n[0], 32LL * 32);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_interp_axis<double, false>), dim3(ew_grid((long long)n[0] * n[1] * 32)), dim3(256), 0, s, t1,
                     E1, (void*)t2, (long long)n[0], 32, n[1], 32LL);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_interp_axis<double, true>), dim3(ew_grid((long long)n[0] * n[1] * n[2])), dim3(256), 0, s, t2,
                     E2, (void*)psi, (long long)n[0] * n[1], 32, n[2], 1LL);
  return hipGetLastError();
}

}  // namespace atus
