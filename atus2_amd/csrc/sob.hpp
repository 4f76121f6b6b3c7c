// sob.hpp -- the kernels of the Sobolev minimiser's loop (CSOB_Base::run).
#pragma once
#include "kernels.hpp"

namespace atus {

// ------------------------------------------------------- the Sobolev loop
// One iteration of CSOB_Base::run on a 2D/3D grid (CSOB_Base.h:431-503).
// With F the unnormalised transform, A = F psi, B = F (W psi) (W = V +
// sum_j g_j |psi_j|^2), phi = alpha k^2, op = 1/(1 + phi) and the transform
// pair's scale s (c = s npts, 1 where dx dk n = 2 pi):
//   psi_sob = F^-1 s op A
//   grad    = F^-1 s op (c phi A + B)     (the filter of -Lap psi + W psi)
//   <psi, grad> = s sum op (c phi |A|^2 + Re A* B),  <psi, psi_sob> = s sum op |A|^2
// so the Laplacian is never formed, both products of the projection come
// from the spectrum, and the projected gradient grad - fak psi_sob needs one
// inverse transform instead of one for each of psi_sob, Lap psi and grad.
// The passes of an iteration, in 16-byte reads and writes per point:
//   k_sob_turn  last axis: inverse, the update of psi, forward of psi and
//               W psi (reads d, psi, V; writes psi, A, B: 5.5)
//   k_pass      middle axis (3D) forward of A and B (4)
//   k_sob_mix   axis 0: forward of A and B, the two combinations above and
//               their products with A (4)
//   k_sob_pull  axis 0: their difference, inverse (3)
//   k_pass      middle axis (3D) inverse (2)
// 18.5 in 3D; the same iteration by its two filters (psi_sob, Lap psi, then
// the gradient through the filter) takes 31.5.  At 128^3 (psi, V and the
// spectra, 112 MiB, stay in the last-level cache) what they stream bounds
// them: an iteration takes 109 us, 5.7 TB/s, against 201 us by the filters.
// At 32^3 their 5 launches of 3.3-6.9 us do: 26 us against 59 us for 14.

struct SobState {
  double f[2];        // scale of psi before this iteration's update (1 or 1/sqrt(N))
  double N[2];        // particle numbers of the current psi
  double res_tot;     // residual of the last iteration performed
  long long iters;    // iterations performed
  int done;           // an iteration ended with res_tot <= eps
  int renorm;         // this iteration renormalises (f != 1)
};
// per performed iteration: N[0], N[1] (checked before its update), whether
// it renormalised, res_tot
constexpr int SOB_LOG_VALS = 4;
constexpr int SOB_MAX_CHUNK = 1024;

// sums of a workgroup of any whole number of wavefronts, returned to every
// thread (fixed order)
template <int NV>
__device__ __forceinline__ void block_sum(double (&acc)[NV]) {
  __shared__ double sh[16][NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc[v] += __shfl_xor(acc[v], off, 64);
  }
  __syncthreads();  // the last use of sh is done
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int v = 0; v < NV; ++v) sh[threadIdx.x >> 6][v] = acc[v];
  }
  __syncthreads();
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    acc[v] = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) acc[v] += sh[w][v];
  }
}

// what advances the loop's state after an update
struct SobFinish {
  const double* part;  // k_sob_turn's partials [nb][2 nw]: |d_i|^2, |psi_i|^2
  int nb;
  int nw;
  double ar, eps;
  int init;            // only N of the current psi (start of a run of iterations)
  double* log;
  int slot;
};

// one workgroup: sums the partials in a fixed order and advances the state.
// Unless the loop is done: res_i = ar sum |d_i|^2 (Compute_res,
// CSOB_Base.h:370-397), res_tot = sqrt(sum res_i^2), the iteration's log
// entry, iters + 1, done if res_tot <= eps; then N of the updated psi and
// the renormalisation of the next iteration (|N_i - 1| > 1e-5 for any i,
// CSOB_Base.h:470-479).
__device__ __forceinline__ void sob_finish(SobState* __restrict__ st, const SobFinish& fin) {
  double tot[4] = {0.0, 0.0, 0.0, 0.0};
  const int nv = 2 * fin.nw;
  for (int b = threadIdx.x; b < fin.nb; b += blockDim.x) {
    tot[0] += fin.part[(long long)b * nv];
    tot[1] += fin.part[(long long)b * nv + 1];
    if (fin.nw > 1) {
      tot[2] += fin.part[(long long)b * nv + 2];
      tot[3] += fin.part[(long long)b * nv + 3];
    }
  }
  block_sum<4>(tot);
  if (threadIdx.x != 0) return;
  if (fin.init) {
    st->done = 0;
    st->iters = 0;
    st->res_tot = 0.0;
  } else {
    if (st->done) return;
    double rsq = 0.0;
    for (int i = 0; i < fin.nw; ++i) {
      const double r = tot[2 * i] * fin.ar;
      rsq += r * r;
    }
    const double rt = sqrt(rsq);
    double* e = fin.log + (long long)fin.slot * SOB_LOG_VALS;
    e[0] = st->N[0];
    e[1] = fin.nw > 1 ? st->N[1] : 0.0;
    e[2] = st->renorm;
    e[3] = rt;
    st->res_tot = rt;
    st->iters += 1;
    if (rt <= fin.eps) st->done = 1;
  }
  bool renorm = false;
  for (int i = 0; i < fin.nw; ++i) {
    st->N[i] = fin.ar * tot[2 * i + 1];
    if (fabs(st->N[i] - 1) > 1e-5) renorm = true;
  }
  for (int i = 0; i < fin.nw; ++i) st->f[i] = renorm ? 1.0 / sqrt(st->N[i]) : 1.0;
  st->renorm = renorm ? 1 : 0;
}

struct SobTurn {
  const double* pot;  // nw x npts
  double gs[4];       // row-major nw x nw
  double step;
  int update;         // 0: the first spectra of a run of iterations
  int forward;        // 0: the last iteration of a run
};

// spec: [2 nw][npts], the projected gradients d_i (transformed along this
// axis only) in the first nw on entry, A_i and B_i on exit.
// psi_i <- f_i psi_i - step d_i unless the loop is done (the update of psi,
// CSOB_Base.h:481-492); partials [workgroup][2 nw]: |d_i|^2 and |psi_i|^2.
template <int N, int RM, int NW>
__global__ __launch_bounds__(256) void k_sob_turn(double2* __restrict__ psi, double2* __restrict__ spec,
                                                  long long npts, AxisGeo g, const double2* __restrict__ tw,
                                                  SobTurn a, const SobState* __restrict__ st,
                                                  double* __restrict__ partials) {
  extern __shared__ double2 lds_all[];
  constexpr int R = Plan<N, RM>::R, P = Plan<N, RM>::P;
  constexpr bool WAVE = P <= 64;
  PencilMap<N, RM, true> m(g);
  double2* lds = lds_all + m.p * g.ls;
  const double2* twl = stage_table<N>(lds_all + (size_t)g.T * g.ls, fft_tw<N, RM>(tw));
  double2 v[NW][R];
#pragma unroll
  for (int c = 0; c < NW; ++c) load_pencil<N, RM>(v[c], psi + c * npts, m.base, 1, m.t, m.valid);
  if constexpr (tables_in_lds<N>()) __syncthreads();
  double acc[2 * NW];
#pragma unroll
  for (int c = 0; c < NW; ++c) {
    acc[2 * c] = 0.0;
    if (a.update) {
      const double f = st->f[c];
      const bool frozen = st->done != 0;
      double2 d[R];
      load_pencil<N, RM>(d, spec + c * npts, m.base, 1, m.t, m.valid);
      fft_pencil<N, RM, +1, WAVE>(d, m.t, lds, fresh_tw<N>(twl));
#pragma unroll
      for (int i = 0; i < R; ++i) {
        acc[2 * c] += d[i].x * d[i].x + d[i].y * d[i].y;
        if (!frozen) {
          if (f != 1.0) v[c][i] = cscale(v[c][i], f);
          v[c][i].x -= a.step * d[i].x;
          v[c][i].y -= a.step * d[i].y;
        }
      }
      if (!frozen) store_pencil<N, RM>(v[c], psi + c * npts, m.base, 1, m.t, m.valid);
    }
    acc[2 * c + 1] = 0.0;
#pragma unroll
    for (int i = 0; i < R; ++i) acc[2 * c + 1] += v[c][i].x * v[c][i].x + v[c][i].y * v[c][i].y;
  }
  block_sum<2 * NW>(acc);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int q = 0; q < 2 * NW; ++q) partials[(long long)blockIdx.x * (2 * NW) + q] = acc[q];
  }
  if (!a.forward) return;
#pragma unroll
  for (int c = 0; c < NW; ++c) {
    double2 w[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
      double W = 0.0;
#pragma unroll
      for (int j = 0; j < NW; ++j) W += a.gs[j + NW * c] * (v[j][i].x * v[j][i].x + v[j][i].y * v[j][i].y);
      if (m.valid) W += a.pot[c * npts + m.base + m.t + P * i];
      w[i] = cscale(v[c][i], W);
    }
    fft_pencil<N, RM, -1, WAVE>(w, m.t, lds, fresh_tw<N>(twl));
    store_pencil<N, RM>(w, spec + (NW + c) * npts, m.base, 1, m.t, m.valid);
  }
#pragma unroll
  for (int c = 0; c < NW; ++c) {
    fft_pencil<N, RM, -1, WAVE>(v[c], m.t, lds, fresh_tw<N>(twl));
    store_pencil<N, RM>(v[c], spec + c * npts, m.base, 1, m.t, m.valid);
  }
}

struct SobMix {
  double alpha[2];
  double dk[3];
  int n[3];
  int dim;
  double s, c;  // the transform pair's scale; s npts
};

// axis 0 of A_i and B_i (blockIdx.y = i): A <- s op (c phi A + B), B <- s op A
// and partials [i][workgroup]: their products with A
template <int N, int RM>
__global__ __launch_bounds__(256) void k_sob_mix(double2* __restrict__ spec, long long npts, int nw, AxisGeo g,
                                                 const double2* __restrict__ tw, SobMix sa,
                                                 double* __restrict__ partials) {
  extern __shared__ double2 lds_all[];
  constexpr int R = Plan<N, RM>::R, P = Plan<N, RM>::P;
  PencilMap<N, RM, false> m(g);
  double2* lds = lds_all + m.p * g.ls;
  const double2* twl = stage_table<N>(lds_all + (size_t)g.T * g.ls, fft_tw<N, RM>(tw));
  double2* A = spec + (long long)blockIdx.y * npts;
  double2* B = A + (long long)nw * npts;
  const double alpha = sa.alpha[blockIdx.y];
  double2 v[R], w[R];
  load_pencil<N, RM>(v, A, m.base, m.stride, m.t, m.valid);
  load_pencil<N, RM>(w, B, m.base, m.stride, m.t, m.valid);
  // alpha k^2 of the other axes
  double phi12 = 0.0;
  {
    const unsigned n2 = sa.dim == 3 ? (unsigned)sa.n[2] : 1u;
    const unsigned col = (unsigned)m.pid;  // one slab: the column index
    const double k1 = kval((int)(col / n2), sa.n[1], sa.dk[1]);
    phi12 = (k1 * alpha) * k1;
    if (sa.dim == 3) {
      const double k2 = kval((int)(col % n2), sa.n[2], sa.dk[2]);
      phi12 += (k2 * alpha) * k2;
    }
  }
  if constexpr (tables_in_lds<N>()) __syncthreads();
  fft_pencil<N, RM, -1, false>(v, m.t, lds, fresh_tw<N>(twl));
  fft_pencil<N, RM, -1, false>(w, m.t, lds, fresh_tw<N>(twl));
  double acc[2] = {0.0, 0.0};
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const double k0 = kval(m.t + P * i, N, sa.dk[0]);
    const double phi = (k0 * alpha) * k0 + phi12;
    const double op = sa.s / (1.0 + phi), cphi = sa.c * phi;
    const double2 a = v[i];
    v[i] = make_double2(op * (cphi * a.x + w[i].x), op * (cphi * a.y + w[i].y));
    w[i] = cscale(a, op);
    acc[0] += a.x * v[i].x + a.y * v[i].y;
    acc[1] += a.x * w[i].x + a.y * w[i].y;
  }
  store_pencil<N, RM>(v, A, m.base, m.stride, m.t, m.valid);
  store_pencil<N, RM>(w, B, m.base, m.stride, m.t, m.valid);
  block_sum<2>(acc);
  if (threadIdx.x == 0) {
    double* o = partials + ((long long)blockIdx.y * gridDim.x + blockIdx.x) * 2;
    o[0] = acc[0];
    o[1] = acc[1];
  }
}

// the projected gradient A - fak B, fak = the ratio of k_sob_mix's products
// (every workgroup sums its nb partials, in the same order), inverse along
// axis 0 into A.  The first workgroup also advances the loop's state after
// the update that made these spectra.
template <int N, int RM>
__global__ __launch_bounds__(256) void k_sob_pull(double2* __restrict__ spec, long long npts, int nw, AxisGeo g,
                                                  const double2* __restrict__ tw, const double* __restrict__ partials,
                                                  int nb, SobState* __restrict__ st, SobFinish fin) {
  extern __shared__ double2 lds_all[];
  constexpr int R = Plan<N, RM>::R;
  PencilMap<N, RM, false> m(g);
  double2* lds = lds_all + m.p * g.ls;
  const double2* twl = stage_table<N>(lds_all + (size_t)g.T * g.ls, fft_tw<N, RM>(tw));
  double2* A = spec + (long long)blockIdx.y * npts;
  double2 v[R], w[R];
  load_pencil<N, RM>(v, A, m.base, m.stride, m.t, m.valid);
  load_pencil<N, RM>(w, A + (long long)nw * npts, m.base, m.stride, m.t, m.valid);
  double pr[2] = {0.0, 0.0};
  const double* p = partials + (long long)blockIdx.y * nb * 2;
  for (int b = threadIdx.x; b < nb; b += blockDim.x) {
    pr[0] += p[2 * b];
    pr[1] += p[2 * b + 1];
  }
  block_sum<2>(pr);  // its barriers also cover the staged twiddles
  const double fak = pr[0] / pr[1];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    v[i].x -= fak * w[i].x;
    v[i].y -= fak * w[i].y;
  }
  fft_pencil<N, RM, +1, false>(v, m.t, lds, fresh_tw<N>(twl));
  store_pencil<N, RM>(v, A, m.base, m.stride, m.t, m.valid);
  if (blockIdx.x == 0 && blockIdx.y == 0) sob_finish(st, fin);
}

// The whole loop of a 1D grid (N <= 4096) in one workgroup: psi stays in
// registers over up to `count` iterations and the kernel returns at the one
// that ends with res_tot <= eps.  An iteration is a serial chain of 3 nw
// transforms and three workgroup sums; latency bounds it, so the pencil takes
// the plan of 8 values per thread, as a resident block's does.  A launch per
// pass (11 per iteration and wave function) had cost about 45 us each
// iteration whatever the length.
template <int N, int RM, int NW, int LB>
__global__ __launch_bounds__(LB) void k_sob_line(double2* __restrict__ psi, AxisGeo g, const double2* __restrict__ tw,
                                                 SobTurn a, SobMix sa, double ar, double eps, int count,
                                                 SobState* __restrict__ st, double* __restrict__ log) {
  extern __shared__ double2 lds_all[];
  constexpr int R = Plan<N, RM>::R, P = Plan<N, RM>::P;
  constexpr bool WAVE = P <= 64;
  PencilMap<N, RM, true> m(g);  // pencil 0; lanes beyond it only fill the wavefront
  double2* lds = lds_all + m.p * g.ls;
  const double2* twl = stage_table<N>(lds_all + (size_t)g.T * g.ls, fft_tw<N, RM>(tw));
  double2 v[NW][R];
#pragma unroll
  for (int c = 0; c < NW; ++c) load_pencil<N, RM>(v[c], psi + c * (long long)N, m.base, 1, m.t, m.valid);
  __syncthreads();
  int it = 0;
  double rt = 0.0;
  bool done = false;
  while (it < count && !done) {
    double nrm[NW];
#pragma unroll
    for (int c = 0; c < NW; ++c) {
      nrm[c] = 0.0;
#pragma unroll
      for (int i = 0; i < R; ++i) nrm[c] += v[c][i].x * v[c][i].x + v[c][i].y * v[c][i].y;
    }
    block_sum<NW>(nrm);
    bool renorm = false;
#pragma unroll
    for (int c = 0; c < NW; ++c) {
      nrm[c] *= ar;
      if (fabs(nrm[c] - 1) > 1e-5) renorm = true;
    }
    double2 d[NW][R];
#pragma unroll
    for (int c = 0; c < NW; ++c) {
      double2 w[R];
#pragma unroll
      for (int i = 0; i < R; ++i) {
        double W = 0.0;
#pragma unroll
        for (int j = 0; j < NW; ++j) W += a.gs[j + NW * c] * (v[j][i].x * v[j][i].x + v[j][i].y * v[j][i].y);
        if (m.valid) W += a.pot[c * (long long)N + m.t + P * i];
        w[i] = cscale(v[c][i], W);
        d[c][i] = v[c][i];
      }
      fft_pencil<N, RM, -1, WAVE>(d[c], m.t, lds, fresh_tw<N>(twl));
      fft_pencil<N, RM, -1, WAVE>(w, m.t, lds, fresh_tw<N>(twl));
      double pr[2] = {0.0, 0.0};
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const double k0 = kval(m.t + P * i, N, sa.dk[0]);
        const double phi = (k0 * sa.alpha[c]) * k0;
        const double op = sa.s / (1.0 + phi), cphi = sa.c * phi;
        const double2 q = d[c][i];
        d[c][i] = make_double2(op * (cphi * q.x + w[i].x), op * (cphi * q.y + w[i].y));
        w[i] = cscale(q, op);
        pr[0] += q.x * d[c][i].x + q.y * d[c][i].y;
        pr[1] += q.x * w[i].x + q.y * w[i].y;
      }
      block_sum<2>(pr);
      const double fak = pr[0] / pr[1];
#pragma unroll
      for (int i = 0; i < R; ++i) {
        d[c][i].x -= fak * w[i].x;
        d[c][i].y -= fak * w[i].y;
      }
      fft_pencil<N, RM, +1, WAVE>(d[c], m.t, lds, fresh_tw<N>(twl));
    }
    double rs[NW];
#pragma unroll
    for (int c = 0; c < NW; ++c) {
      rs[c] = 0.0;
      const double f = renorm ? 1.0 / sqrt(nrm[c]) : 1.0;
#pragma unroll
      for (int i = 0; i < R; ++i) {
        rs[c] += d[c][i].x * d[c][i].x + d[c][i].y * d[c][i].y;
        if (renorm) v[c][i] = cscale(v[c][i], f);
        v[c][i].x -= a.step * d[c][i].x;
        v[c][i].y -= a.step * d[c][i].y;
      }
    }
    block_sum<NW>(rs);
    double rsq = 0.0;
#pragma unroll
    for (int c = 0; c < NW; ++c) rsq += (rs[c] * ar) * (rs[c] * ar);
    rt = sqrt(rsq);
    done = rt <= eps;
    if (threadIdx.x == 0) {
      double* e = log + (long long)it * SOB_LOG_VALS;
      e[0] = nrm[0];
      e[1] = NW > 1 ? nrm[NW - 1] : 0.0;
      e[2] = renorm ? 1.0 : 0.0;
      e[3] = rt;
    }
    ++it;
  }
#pragma unroll
  for (int c = 0; c < NW; ++c) store_pencil<N, RM>(v[c], psi + c * (long long)N, m.base, 1, m.t, m.valid);
  if (threadIdx.x == 0) {
    st->iters = it;
    st->res_tot = rt;
    st->done = done ? 1 : 0;
  }
}

}  // namespace atus
