// kernels_misc.hpp -- non-template kernels, launched only by atus_abi.hip
// (kept out of kernels.hpp so each has one definition).
#pragma once
#include "kernels.hpp"
#include "sob.hpp"

namespace atus {

// psi *= exp(i p.x)  (CRT_Base::Setup_Momentum, CRT_Base.h:449-473)
__global__ __launch_bounds__(256) void k_momentum(double2* __restrict__ psi, Grid gr, double p0, double p1,
                                                  double p2) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long l = (long long)blockIdx.x * blockDim.x + threadIdx.x; l < gr.npts; l += stride) {
    int id[3];
    split_point(l, gr, id);
    const int i0 = id[0], i1 = id[1], i2 = id[2];
    double px = p0 * ((double)(i0 - gr.n[0] / 2) * gr.dx[0]);
    if (gr.dim > 1) px += p1 * ((double)(i1 - gr.n[1] / 2) * gr.dx[1]);
    if (gr.dim > 2) px += p2 * ((double)(i2 - gr.n[2] / 2) * gr.dx[2]);
    double s, c;
    sincos(px, &s, &c);
    const double2 a = psi[l];
    psi[l] = make_double2(a.x * c - a.y * s, a.x * s + a.y * c);
  }
}

// inflate_domain (inflate_domain.cpp:41-223) on the device, one thread per
// destination point of one component (blockIdx.y): FIX == false pads the
// source grid, fak times smaller per axis, with zeros around the centre
// (offset (n_dst - n_src)/2); FIX == true keeps the number of points and
// places every fak-th source point around the centre (offset
// n*(fak-1)/2/fak); everything else is zero
template <bool FIX>
__global__ __launch_bounds__(256) void k_inflate(const double2* __restrict__ src, double2* __restrict__ dst, Grid gs,
                                                 Grid gd, int fak, long long src_stride, long long dst_stride) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  const double2* s = src + (long long)blockIdx.y * src_stride;
  double2* d = dst + (long long)blockIdx.y * dst_stride;
  for (long long l = (long long)blockIdx.x * blockDim.x + threadIdx.x; l < gd.npts; l += stride) {
    int id[3];
    split_point(l, gd, id);
    bool inside = true;
    long long ls = 0;
    for (int a = 0; a < 3; ++a) {
      int is;
      if (!FIX) {
        is = id[a] - (gd.n[a] - gs.n[a]) / 2;
      } else {
        // destination off + i/fak <- source i for i = 0, fak, 2 fak, ...
        const int off = gs.n[a] * (fak - 1) / 2 / fak;
        const int q = id[a] - off;
        is = q * fak;
        if (gs.n[a] == 1) is = q;  // unused axis
      }
      if (is < 0 || is >= gs.n[a]) inside = false;
      ls = ls * gs.n[a] + (inside ? is : 0);
    }
    d[l] = inside ? s[ls] : make_double2(0.0, 0.0);
  }
}

// streaming copy (bandwidth probe)
__global__ __launch_bounds__(256) void k_copy(const double2* __restrict__ src, double2* __restrict__ dst, long long n) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long l = (long long)blockIdx.x * blockDim.x + threadIdx.x; l < n; l += stride) dst[l] = src[l];
}

// ------------------------------------------------------------ Sobolev loop

// the loop's state after the last update of a run of iterations (after the
// others the next iteration's k_sob_pull advances it)
__global__ __launch_bounds__(RED_THREADS) void k_sob_finish(SobState* __restrict__ st, SobFinish fin) {
  sob_finish(st, fin);
}

__global__ __launch_bounds__(256) void k_scale(double2* __restrict__ psi, long long n, double f) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long l = (long long)blockIdx.x * blockDim.x + threadIdx.x; l < n; l += stride) psi[l] = cscale(psi[l], f);
}


// dst = scale * transpose(src) for `ncomp` matrices of rows x cols, each
// comp_stride elements apart in both buffers; 32 x 32 tiles through LDS,
// one tile per workgroup (blockIdx.x = (comp * row_tiles + i) * col_tiles + j)
__global__ __launch_bounds__(256) void k_transpose(const double2* __restrict__ src, double2* __restrict__ dst,
                                                   long long rows, long long cols, long long comp_stride,
                                                   double scale) {
  __shared__ double2 tile[32][33];
  const long long ct = (cols + 31) / 32, rt = (rows + 31) / 32;
  const long long b = blockIdx.x;
  const long long comp = b / (rt * ct), rem = b % (rt * ct);
  const long long i0 = (rem / ct) * 32, j0 = (rem % ct) * 32;
  src += comp * comp_stride;
  dst += comp * comp_stride;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int k = ty; k < 32; k += 8) {
    const long long i = i0 + k, j = j0 + tx;
    if (i < rows && j < cols) tile[k][tx] = src[i * cols + j];
  }
  __syncthreads();
  for (int k = ty; k < 32; k += 8) {
    const long long j = j0 + k, i = i0 + tx;
    if (i < rows && j < cols) {
      const double2 a = tile[tx][k];
      dst[j * rows + i] = make_double2(a.x * scale, a.y * scale);
    }
  }
}

}  // namespace atus
