// marg.hpp -- densities of a state along one axis, in x and in k space.
#pragma once
#include "launch.hpp"

namespace atus {

// For one axis of N points: (sum of |psi|^2, sum of |F psi|^2) over all other
// coordinates, for every index j of that axis, F the unnormalised transform
// along that axis alone.  By Parseval's theorem the other axes' transforms
// only multiply the second sum by their lengths, so moments of the momentum
// distribution and the kinetic energy need one read of the state per axis,
// where the whole transform and a sum over it take three passes that also
// write (256^3: 82 us each) and a read.
// Workgroups run over the tiles blockIdx.x, + gridDim.x, ...; a thread keeps
// the sums of its elements in registers, the workgroup's pencils are summed
// in LDS, part[blockIdx.x][N] receives the result.  PHASE (last axis): also
// the sum of atan2(Im psi, Re psi) |psi|^2, phase[blockIdx.x].
template <int N, int RM, bool CONTIG, bool PHASE>
__global__ __launch_bounds__(256) void k_marginal(const double2* __restrict__ psi, AxisGeo g,
                                                  const double2* __restrict__ tw, double2* __restrict__ part,
                                                  double* __restrict__ phase) {
  extern __shared__ double2 lds_all[];
  constexpr int R = Plan<N, RM>::R, P = Plan<N, RM>::P;
  constexpr bool WAVE = CONTIG && (P <= 64);
  const double2* twl = stage_table<N>(lds_all + (size_t)g.T * g.ls, fft_tw<N, RM>(tw));
  const int p = CONTIG ? threadIdx.x / P : threadIdx.x % g.T;
  const int t = CONTIG ? threadIdx.x % P : threadIdx.x / g.T;
  double2* lds = lds_all + p * g.ls;
  double ax[R], ak[R], ph = 0.0;
#pragma unroll
  for (int i = 0; i < R; ++i) ax[i] = ak[i] = 0.0;
  if constexpr (tables_in_lds<N>()) __syncthreads();
  for (long long tile = blockIdx.x; tile < g.ntiles; tile += gridDim.x) {
    long long base, stride;
    bool valid;
    if constexpr (CONTIG) {
      const long long pid = tile * g.T + p;
      valid = pid < g.outer;
      base = pid * N;
      stride = 1;
    } else {
      const unsigned o = (unsigned)tile / (unsigned)g.col_tiles;
      const long long col = (long long)((unsigned)tile - o * (unsigned)g.col_tiles) * g.T + p;
      valid = col < g.inner;
      base = (long long)o * N * g.inner + col;
      stride = g.inner;
    }
    double2 v[R];
    load_pencil<N, RM>(v, psi, base, stride, t, valid);
    double phi = 0.0;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const double d = v[i].x * v[i].x + v[i].y * v[i].y;
      ax[i] += d;
      if constexpr (PHASE) phi += atan2(v[i].y, v[i].x) * d;
    }
    if constexpr (PHASE) ph += phi;
    fft_pencil<N, RM, -1, WAVE>(v, t, lds, fresh_tw<N>(twl));
#pragma unroll
    for (int i = 0; i < R; ++i) ak[i] += v[i].x * v[i].x + v[i].y * v[i].y;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < R; ++i) lds[t + P * i] = make_double2(ax[i], ak[i]);
  __syncthreads();
  for (int j = threadIdx.x; j < N; j += blockDim.x) {
    double2 s = lds_all[j];
    for (int q = 1; q < g.T; ++q) s = cadd(s, lds_all[q * g.ls + j]);
    part[(long long)blockIdx.x * N + j] = s;
  }
  if constexpr (PHASE) {
    __syncthreads();
    double* sh = reinterpret_cast<double*>(lds_all);
    sh[threadIdx.x] = ph;
    __syncthreads();
    // contiguous pencils: a power of two of threads
    for (int h = (int)blockDim.x >> 1; h > 0; h >>= 1) {
      if ((int)threadIdx.x < h) sh[threadIdx.x] += sh[threadIdx.x + h];
      __syncthreads();
    }
    if (threadIdx.x == 0) phase[blockIdx.x] = sh[0];
  }
}

// out[j] = sum over nb of part[b][j], j < N, in a fixed order: 16 elements
// per workgroup, 16 threads each
__global__ __launch_bounds__(256) void k_marginal_sum(const double2* __restrict__ part, int nb, int N,
                                                      double2* __restrict__ out) {
  __shared__ double2 sh[16][16];
  const int e = threadIdx.x & 15, q = threadIdx.x >> 4;
  const int j = blockIdx.x * 16 + e;
  double2 s = make_double2(0.0, 0.0);
  if (j < N) {
    // 8 loads in flight: one after another they took 12 us of 512 partials
    int b = q;
    for (; b + 112 < nb; b += 128) {
      double2 w[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) w[i] = part[(long long)(b + 16 * i) * N + j];
#pragma unroll
      for (int i = 0; i < 8; ++i) s = cadd(s, w[i]);
    }
    for (; b < nb; b += 16) s = cadd(s, part[(long long)b * N + j]);
  }
  sh[q][e] = s;
  __syncthreads();
  if (q == 0 && j < N) {
    for (int r = 1; r < 16; ++r) s = cadd(s, sh[r][e]);
    out[j] = s;
  }
}

}  // namespace atus
