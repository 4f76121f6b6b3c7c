// multi.hpp -- V-step kernels of several coupled components, the components
// side by side in one workgroup: thread group c transforms component c, and
// at the V step the groups meet in LDS, where each takes its share of the
// points with all components of each.  No thread holds more than one
// component's values through a transform, and the chain of a step is one
// transform pair and 1/NC of the V step long, not NC pairs and all of it.
#pragma once
#include "launch.hpp"

namespace atus {

// values per thread of a workgroup with all components of a pencil, or 0
// where it would be larger than `most` threads
__host__ __device__ constexpr int comp_rm(int N, int NC, int most) {
  if (N <= 8) return 8;
  if (NC * (N / 8) <= most) return 8;
  return (N >= 32 && NC * (N / 16) <= most) ? 16 : 0;
}

__device__ __forceinline__ double2 sel(bool b, double2 x, double2 y) {
  return make_double2(b ? x.x : y.x, b ? x.y : y.y);
}

// The V step of one pencil held by NC thread groups (group c: component c,
// element t + P i in register i).  region: the pencil's LDS regions, `cs`
// elements apart per component; point(a, j): the step on element j.
// Two components: group 0 takes the lower half of the registers' elements,
// group 1 the upper, so only the halves of the other component cross.
template <int N, int RM, int NC, bool WAVE, class F>
__device__ __forceinline__ void comp_vstep(double2 (&v)[(Plan<N, RM>::R)], int c, int t, double2* region, int cs,
                                           bool valid, const F& point) {
  constexpr int R = Plan<N, RM>::R, P = Plan<N, RM>::P;
  double2* mine = region + c * cs;
  lds_sync<WAVE>();  // the last exchange's reads of the region are done
  if constexpr (NC == 2 && R % 2 == 0) {
    constexpr int H = R / 2;
    double2* peer = region + (1 - c) * cs;
    double2 own[H], oth[H];
#pragma unroll
    for (int k = 0; k < H; ++k) {
      own[k] = sel(c == 0, v[k], v[H + k]);
      oth[k] = sel(c == 0, v[H + k], v[k]);
    }
    const int jown = t + (c == 0 ? 0 : P * H), joth = t + (c == 0 ? P * H : 0);
#pragma unroll
    for (int k = 0; k < H; ++k) mine[lds_pos(joth + P * k)] = oth[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < H; ++k) {
      const int j = jown + P * k;
      const double2 b = peer[lds_pos(j)];
      double2 a[2];
      a[0] = sel(c == 0, own[k], b);
      a[1] = sel(c == 0, b, own[k]);
      if (valid) point(a, j);
      own[k] = sel(c == 0, a[0], a[1]);
      peer[lds_pos(j)] = sel(c == 0, a[1], a[0]);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < H; ++k) {
      oth[k] = mine[lds_pos(joth + P * k)];
      v[k] = sel(c == 0, own[k], oth[k]);
      v[H + k] = sel(c == 0, oth[k], own[k]);
    }
  } else {
#pragma unroll
    for (int i = 0; i < R; ++i) mine[lds_pos(t + P * i)] = v[i];
    __syncthreads();
    if (valid) {
      for (int j = c * P + t; j < N; j += NC * P) {
        double2 a[NC];
#pragma unroll
        for (int q = 0; q < NC; ++q) a[q] = region[q * cs + lds_pos(j)];
        point(a, j);
#pragma unroll
        for (int q = 0; q < NC; ++q) region[q * cs + lds_pos(j)] = a[q];
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < R; ++i) v[i] = mine[lds_pos(t + P * i)];
  }
}

// inverse DFT along the last axis of a 2D/3D grid, V step, forward DFT.
// Workgroup: g.T pencils of NC x P threads.  BATCH: the pencils of all runs
// of a batch, each with its run's parameters.  Against k_vfuse, which holds
// both components of a pencil in the same threads (144 registers, three
// waves per SIMD; here 112, four), a Bragg step takes 12.7 us for 15.6 at
// 128^2, 23.6 for 27.3 at 512^2, 28.6 for 31.2 at 64^3, 103.9 for 108.5 at
// 128^3; between the other stream's passes of a slab chain (256^3) the two
// are equal.
template <int N, int RM, int VK, int NC, bool BATCH, int LB>
__global__ __launch_bounds__(LB) void k_vcomp(double2* __restrict__ psi, long long comp_stride, AxisGeo g,
                                              const double2* __restrict__ tw, VArgs va, VGeo geo) {
  extern __shared__ double2 lds_all[];
  constexpr int P = Plan<N, RM>::P, R = Plan<N, RM>::R;
  constexpr bool WAVE = P <= 64;
  const int q = threadIdx.x / P, t = threadIdx.x % P;
  const int c = q / g.T, p = q % g.T;
  const long long pid = xcd_tile(blockIdx.x, gridDim.x) * g.T + p;
  const bool valid = pid < g.outer;
  double2* region = lds_all + p * g.ls;
  const int cs = g.T * g.ls;
  const double2* twl = stage_table<N>(lds_all + (size_t)NC * cs, fft_tw<N, RM>(tw));
  long long own = pid;  // pencil of its run
  if constexpr (BATCH) {
    const long long r = pid / va.pencils_per_run;
    own = pid - r * va.pencils_per_run;
    if (valid) bind_run(va, r);
    psi += r * va.run_shift;
  }
  double2 v[R];
  load_pencil<N, RM>(v, psi + c * comp_stride, pid * N, 1, t, valid);
  const unsigned ppx = geo.dim == 3 ? (unsigned)geo.n[1] : 1u;
  const int i0 = (int)((unsigned)own / ppx), i1 = (int)((unsigned)own % ppx);
  const double x0 = (double)(i0 - geo.n[0] / 2) * geo.dx[0];
  const auto field = v_field<VK, NC, false>(x0, va);
  if constexpr (tables_in_lds<N>()) __syncthreads();
  fft_pencil<N, RM, +1, WAVE>(v, t, region + c * cs, fresh_tw<N>(twl));
  comp_vstep<N, RM, NC, WAVE>(v, c, t, region, cs, valid, [&](double2(&a)[NC], int j) {
    double bx = 0.0;
    if constexpr (VK == V_DBRAGG || VK == V_NUM_BRAGG || VK == V_RAMAN) {
      // summed over the axes as beta_dot_x does
      bx += va.beta[0] * x0;
      if (geo.dim == 3) bx += va.beta[1] * ((double)(i1 - geo.n[1] / 2) * geo.dx[1]);
      const int last = geo.dim - 1;
      bx += va.beta[last] * ((double)(j - N / 2) * geo.dx[last]);
    }
    any_point<VK, NC, false>(a, x0, bx, pid * N + j, field, va);
  });
  fft_pencil<N, RM, -1, WAVE>(v, t, region + c * cs, fresh_tw<N>(twl));
  store_pencil<N, RM>(v, psi + c * comp_stride, pid * N, 1, t, valid);
}

// whether the twiddles of a resident block fit LDS beside NC regions
template <int N, int NC>
constexpr bool block_tw_in_lds() {
  return (NC + 1) * N <= 9600;
}

// A whole block of 1D runs of NC components in one launch (k_block1d for
// several components): half kinetic, (V, full) x (Nk - 1), V, half.  One
// workgroup holds g.T runs; a thread keeps the 8 full-step phases of its
// elements in registers unless its workgroup is too large for that.
template <int N, int RM, int VK, int NC, bool BATCH, int LB>
__global__ __launch_bounds__(LB) void k_bcomp(double2* __restrict__ psi, long long comp_stride, AxisGeo g,
                                              const double2* __restrict__ tw, BlockPhases ph, VArgs va,
                                              BlockSteps st, double dx0) {
  extern __shared__ double2 lds_all[];
  constexpr int P = Plan<N, RM>::P, R = Plan<N, RM>::R;
  constexpr bool WAVE = P <= 64, KT = block_tw_in_lds<N, NC>();
  constexpr bool KEEP = LB <= 512 && R <= 8;
  const int q = threadIdx.x / P, t = threadIdx.x % P;
  const int c = q / g.T, p = q % g.T;
  const long long run = (long long)blockIdx.x * g.T + p;
  const bool valid = run < g.outer;
  double2* region = lds_all + p * g.ls;
  double2* mine = region + c * g.T * g.ls;
  const int cs = g.T * g.ls;
  const double2* twl = stage_table<N, KT>(lds_all + (size_t)NC * cs, fft_tw<N, RM>(tw));
  const bool sp2 = c >= ph.split;
  const double2* eh = sp2 ? ph.half[1] : ph.half[0];
  const double2* ef = sp2 ? ph.full[1] : ph.full[0];
  // this component's elements of the whole state
  const long long base = (BATCH ? run * NC : 0) * comp_stride + c * comp_stride;
  double2 v[R];
  load_pencil<N, RM>(v, psi, base, 1, t, valid);
  double2 keep[KEEP ? R : 1];
  auto set_phases = [&](const double2* e) {
    if constexpr (KEEP) {
#pragma unroll
      for (int i = 0; i < R; ++i) keep[i] = e[t + P * i];
    }
  };
  set_phases(eh);
  // one component: the potential is the same for every step, read once
  constexpr bool POT = NC == 1 && VK == V_NL;
  double pot[POT ? R : 1];
  if constexpr (POT) {
#pragma unroll
    for (int i = 0; i < R; ++i) pot[i] = (va.pot && valid) ? va.pot[t + P * i] : 0.0;
  }
  __syncthreads();
  // `u` is t again for every step, hidden from the compiler: what follows
  // from it (addresses, coordinates, the run's parameters) is formed anew
  // inside the step instead of being kept in registers across the transforms
  auto kinetic = [&](const double2* eg, int u) {
    double2 e[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if constexpr (KEEP) e[i] = keep[i];
      else e[i] = eg[u + P * i];
    }
    fft_pencil<N, RM, -1, WAVE>(v, u, mine, fresh_tw<N, KT>(twl));
#pragma unroll
    for (int i = 0; i < R; ++i) v[i] = cmul(v[i], e[i]);
    fft_pencil<N, RM, +1, WAVE>(v, u, mine, fresh_tw<N, KT>(twl));
  };
  kinetic(eh, t);
  set_phases(ef);
  for (int s = 0; s < st.Nk; ++s) {
    int u = t;
    asm volatile("" : "+v"(u));
    va.t1 = st.t1[s];
    if constexpr (BATCH) {
      va.Fm = st.F + (size_t)s * g.outer;
      long long r = run;
      asm volatile("" : "+v"(r));
      if (valid) bind_run(va, r);
    } else {
      va.F = st.F[s];
    }
    if constexpr (NC == 1) {
#pragma unroll
      for (int i = 0; i < R; ++i) {
        double2 a[1] = {v[i]};
        if constexpr (POT) {
          const double extra[1] = {pot[i]};
          nl_point<1, true, true>(a, extra, va);
        } else {
          any_point<VK, 1, true>(a, (double)(u + P * i - N / 2) * dx0, 0.0, u + P * i, NoField{}, va);
        }
        v[i] = a[0];
      }
    } else {
      comp_vstep<N, RM, NC, WAVE>(v, c, u, region, cs, valid, [&](double2(&a)[NC], int j) {
        const double x0 = (double)(j - N / 2) * dx0;
        any_point<VK, NC, true>(a, x0, 0.0, j, v_field<VK, NC, true>(x0, va), va);
      });
    }
    const bool last = s + 1 == st.Nk;
    if (last) set_phases(eh);
    kinetic(last ? eh : ef, u);
  }
  store_pencil<N, RM>(v, psi, base, 1, t, valid);
}

}  // namespace atus
