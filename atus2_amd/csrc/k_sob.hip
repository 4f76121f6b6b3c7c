// k_sob.hip -- the Sobolev passes and the pointwise V launcher.
#include "launch.hpp"
#include "sob.hpp"

namespace atus {

// The passes of an iteration hold two spectra per thread, so they take the
// plan of 8 values wherever the contiguous pencil fits a workgroup with it.
template <int N>
constexpr int sob_rm() {
  return (N > 8 && N / 8 <= 256) ? 8 : 16;
}

template <int N, int NW>
static hipError_t turn_go(double2* psi, double2* spec, long long npts, const double2* tw, const SobTurn& a,
                          const SobState* st, double* partials, unsigned* nblocks, const Limits& lim, hipStream_t s) {
  constexpr int RM = sob_rm<N>();
  PassCfg c = make_pass_cfg(N, RM, 1, npts / N, 1, lim);
  if (c.block.x == 0 || c.block.x > 256 || c.grid.x == 0) return hipErrorInvalidConfiguration;
  *nblocks = c.grid.x;
  if (!partials) return hipSuccess;
  static bool ok = false;
  hipError_t e = allow_lds(k_sob_turn<N, RM, NW>, c.lds, ok);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_sob_turn<N, RM, NW>), c.grid, c.block, c.lds, s, psi, spec, npts, c.g, tw, a, st, partials);
  return hipGetLastError();
}

hipError_t launch_sob_turn(int N, int nw, double2* psi, double2* spec, long long npts, const double2* tw,
                           const SobTurn& a, const SobState* st, double* partials, unsigned* nblocks,
                           const Limits& lim, hipStream_t s) {
  if (nw != 1 && nw != 2) return hipErrorInvalidValue;
  switch (N) {
#define ATUS_CASE(n)                                                                              \
  case n:                                                                                         \
    return nw == 1 ? turn_go<n, 1>(psi, spec, npts, tw, a, st, partials, nblocks, lim, s)         \
                   : turn_go<n, 2>(psi, spec, npts, tw, a, st, partials, nblocks, lim, s);
    ATUS_CASE(2) ATUS_CASE(4) ATUS_CASE(8) ATUS_CASE(16) ATUS_CASE(32) ATUS_CASE(64) ATUS_CASE(128)
    ATUS_CASE(256) ATUS_CASE(512) ATUS_CASE(1024) ATUS_CASE(2048) ATUS_CASE(4096)
#undef ATUS_CASE
    default: return hipErrorInvalidValue;
  }
}

// axis 0, nw components; whole wavefronts also where the columns are fewer
template <int N>
static PassCfg sob_axis0_cfg(int nw, long long inner, const Limits& lim) {
  return make_pass_cfg(N, sob_rm<N>(), inner, 1, nw, lim, 1, 256, -1, 64);
}

template <int N>
static hipError_t mix_go(int nw, double2* spec, long long npts, long long inner, const double2* tw, const SobMix& sa,
                         double* partials, unsigned* nblocks, const Limits& lim, hipStream_t s) {
  PassCfg c = sob_axis0_cfg<N>(nw, inner, lim);
  if (c.block.x == 0 || c.block.x > 256 || c.grid.x == 0) return hipErrorInvalidConfiguration;
  *nblocks = c.grid.x;
  if (!partials) return hipSuccess;
  static bool ok = false;
  hipError_t e = allow_lds(k_sob_mix<N, sob_rm<N>()>, c.lds, ok);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_sob_mix<N, sob_rm<N>()>), c.grid, c.block, c.lds, s, spec, npts, nw, c.g, tw, sa, partials);
  return hipGetLastError();
}

template <int N>
static hipError_t pull_go(int nw, double2* spec, long long npts, long long inner, const double2* tw,
                          const double* partials, int nb, SobState* st, const SobFinish& fin, const Limits& lim,
                          hipStream_t s) {
  PassCfg c = sob_axis0_cfg<N>(nw, inner, lim);
  if (c.block.x == 0 || c.block.x > 256 || c.grid.x == 0) return hipErrorInvalidConfiguration;
  static bool ok = false;
  hipError_t e = allow_lds(k_sob_pull<N, sob_rm<N>()>, c.lds, ok);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_sob_pull<N, sob_rm<N>()>), c.grid, c.block, c.lds, s, spec, npts, nw, c.g, tw, partials, nb, st,
                     fin);
  return hipGetLastError();
}

hipError_t launch_sob_mix(int N, int nw, double2* spec, long long npts, long long inner, const double2* tw,
                          const SobMix& sa, double* partials, unsigned* nblocks, const Limits& lim, hipStream_t s) {
  switch (N) {
#define ATUS_CASE(n) \
  case n: return mix_go<n>(nw, spec, npts, inner, tw, sa, partials, nblocks, lim, s);
    ATUS_CASE(2) ATUS_CASE(4) ATUS_CASE(8) ATUS_CASE(16) ATUS_CASE(32) ATUS_CASE(64) ATUS_CASE(128)
    ATUS_CASE(256) ATUS_CASE(512) ATUS_CASE(1024) ATUS_CASE(2048) ATUS_CASE(4096)
#undef ATUS_CASE
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_sob_pull(int N, int nw, double2* spec, long long npts, long long inner, const double2* tw,
                           const double* partials, int nb, SobState* st, const SobFinish& fin, const Limits& lim,
                           hipStream_t s) {
  switch (N) {
#define ATUS_CASE(n) \
  case n: return pull_go<n>(nw, spec, npts, inner, tw, partials, nb, st, fin, lim, s);
    ATUS_CASE(2) ATUS_CASE(4) ATUS_CASE(8) ATUS_CASE(16) ATUS_CASE(32) ATUS_CASE(64) ATUS_CASE(128)
    ATUS_CASE(256) ATUS_CASE(512) ATUS_CASE(1024) ATUS_CASE(2048) ATUS_CASE(4096)
#undef ATUS_CASE
    default: return hipErrorInvalidValue;
  }
}

template <int N, int NW>
static hipError_t line_go(double2* psi, const double2* tw, const SobTurn& a, const SobMix& sa, double ar, double eps,
                          int count, SobState* st, double* log, const Limits& lim, hipStream_t s) {
  constexpr int RM = N > 8 ? 8 : 16, P = Plan<N, RM>::P;
  // one pencil, in whole wavefronts (the spare lanes hold invalid pencils)
  constexpr int LB = P > 64 ? P : 64;
  PassCfg c = make_pass_cfg(N, RM, 1, 1, 1, lim.lds, 1, LB);
  if (c.block.x != (unsigned)LB || c.grid.x != 1) return hipErrorInvalidConfiguration;
  static bool ok = false;
  hipError_t e = allow_lds(k_sob_line<N, RM, NW, LB>, c.lds, ok);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_sob_line<N, RM, NW, LB>), c.grid, c.block, c.lds, s, psi, c.g, tw, a, sa, ar, eps, count, st,
                     log);
  return hipGetLastError();
}

hipError_t launch_sob_line(int N, int nw, double2* psi, const double2* tw, const SobTurn& a, const SobMix& sa,
                           double ar, double eps, int count, SobState* st, double* log, const Limits& lim,
                           hipStream_t s) {
  if (nw != 1 && nw != 2) return hipErrorInvalidValue;
  switch (N) {
#define ATUS_CASE(n)                                                                  \
  case n:                                                                             \
    return nw == 1 ? line_go<n, 1>(psi, tw, a, sa, ar, eps, count, st, log, lim, s)   \
                   : line_go<n, 2>(psi, tw, a, sa, ar, eps, count, st, log, lim, s);
    ATUS_CASE(2) ATUS_CASE(4) ATUS_CASE(8) ATUS_CASE(16) ATUS_CASE(32) ATUS_CASE(64) ATUS_CASE(128)
    ATUS_CASE(256) ATUS_CASE(512) ATUS_CASE(1024) ATUS_CASE(2048) ATUS_CASE(4096)
#undef ATUS_CASE
    default: return hipErrorInvalidValue;
  }
}

static unsigned point_blocks(long long n) {
  long long b = (n + 255) / 256;
  if (b > 8192) b = 8192;
  if (b < 1) b = 1;
  return (unsigned)b;
}

hipError_t launch_point(int vk, int nc, double2* psi, const Grid& gr, const VArgs& va, hipStream_t s) {
  dim3 grid(point_blocks(gr.npts)), block(256);
#define ATUS_PT(V, C) \
  if (vk == V && nc == C) { hipLaunchKernelGGL((k_point<V, C>), grid, block, 0, s, psi, gr, va); return hipGetLastError(); }
  ATUS_PT(V_NL, 1) ATUS_PT(V_NL, 2) ATUS_PT(V_NL, 3) ATUS_PT(V_NL, 4)
  ATUS_PT(V_NL_IF, 1) ATUS_PT(V_NL_IF, 2) ATUS_PT(V_NL_IF, 3) ATUS_PT(V_NL_IF, 4)
  ATUS_PT(V_BRAGG, 2)
  ATUS_PT(V_NL_IF2, 2) ATUS_PT(V_NL_IF2, 4) ATUS_PT(V_BRAGG_DS, 4)
  ATUS_PT(V_DBRAGG, 3) ATUS_PT(V_NUM_BRAGG, 2) ATUS_PT(V_NUM_BRAGG, 3) ATUS_PT(V_RAMAN, 3) ATUS_PT(V_RAMAN, 4)
#undef ATUS_PT
  return hipErrorInvalidValue;
}

}  // namespace atus
