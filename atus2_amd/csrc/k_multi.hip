// k_multi.hip -- the multi-component V passes and resident 1D blocks.
#include "multi.hpp"

namespace atus {

// workgroup shape of T pencils x NC thread groups: make_pass_cfg's tile for
// one component, times NC
static PassCfg comp_cfg(int N, int rm, int nc, long long pencils, const Limits& lim, int most, bool tw_lds) {
  const int P = threads_per_pencil(N, rm);
  // about 256 threads, at least one pencil
  int cap = 256;
  while (cap > P && cap * nc > 256) cap >>= 1;
  if (cap < P) cap = P;
  const size_t tw = tw_lds ? (size_t)N * sizeof(double2) : 0;
  const size_t each = lim.lds > tw ? (lim.lds - tw) / nc : 0;
  PassCfg c = make_pass_cfg(N, rm, 1, pencils, nc, Limits{each, lim.threads}, 0, cap, 0);
  if (c.block.x == 0 || (int)(c.block.x * nc) > most) {
    c.block = dim3(0);
    return c;
  }
  c.block = dim3(c.block.x * nc);
  c.grid = dim3(c.grid.x);
  c.lds = c.lds * nc + tw;
  return c;
}

// ------------------------------------------------ the pass along the last axis

constexpr int VCOMP_MOST = 512;  // threads per workgroup

template <int N, int VK, int NC, bool BATCH>
static hipError_t vcomp_go(double2* psi, long long cs, long long outer, const double2* tw, const VArgs& va,
                           const VGeo& geo, const Limits& lim, hipStream_t s) {
  constexpr int RM = comp_rm(N, NC, VCOMP_MOST);
  if constexpr (RM != 8) {
    return hipErrorInvalidValue;
  } else {
    constexpr int LB = NC * Plan<N, RM>::P <= 256 ? 256 : 512;
    PassCfg c = comp_cfg(N, RM, NC, outer, lim, LB, tables_in_lds<N>());
    if (c.block.x == 0 || c.grid.x == 0) return hipErrorInvalidConfiguration;
    static bool ok = false;
    hipError_t e = allow_lds(k_vcomp<N, RM, VK, NC, BATCH, LB>, c.lds, ok);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_vcomp<N, RM, VK, NC, BATCH, LB>), c.grid, c.block, c.lds, s, psi, cs, c.g, tw, va, geo);
    return hipGetLastError();
  }
}

#define ATUS_COMP_KINDS(X)                                                                                        \
  X(V_NL, 2) X(V_NL_IF, 2) X(V_BRAGG, 2) X(V_NL_IF2, 2) X(V_NUM_BRAGG, 2) X(V_NL, 3) X(V_NL_IF, 3) X(V_DBRAGG, 3) \
  X(V_NUM_BRAGG, 3) X(V_RAMAN, 3) X(V_NL, 4) X(V_NL_IF, 4) X(V_NL_IF2, 4) X(V_BRAGG_DS, 4) X(V_RAMAN, 4)

bool vcomp_ok(int N, int vk, int nc) {
  if (comp_rm(N, nc, VCOMP_MOST) != 8) return false;
#define ATUS_K(V, C) \
  if (vk == V && nc == C) return true;
  ATUS_COMP_KINDS(ATUS_K)
#undef ATUS_K
  return false;
}

hipError_t launch_vcomp(int N, int vk, int nc, bool batch, double2* psi, long long comp_stride, long long outer,
                        const double2* tw, const VArgs& va, const VGeo& geo, const Limits& lim, hipStream_t s) {
#define ATUS_K(V, C) \
  if (!batch && vk == V && nc == C) return vcomp_go<ATUS_N, V, C, false>(psi, comp_stride, outer, tw, va, geo, lim, s);
  switch (N) {
#define ATUS_CASE(n)               \
  case n: {                        \
    constexpr int ATUS_N = n;      \
    if (batch && nc == 2 && vk == V_BRAGG) return vcomp_go<n, V_BRAGG, 2, true>(psi, comp_stride, outer, tw, va, geo, lim, s); \
    if (batch && nc == 2 && vk == V_NL_IF) return vcomp_go<n, V_NL_IF, 2, true>(psi, comp_stride, outer, tw, va, geo, lim, s); \
    ATUS_COMP_KINDS(ATUS_K) break; \
  }
    ATUS_CASE(2) ATUS_CASE(4) ATUS_CASE(8) ATUS_CASE(16) ATUS_CASE(32) ATUS_CASE(64) ATUS_CASE(128)
    ATUS_CASE(256) ATUS_CASE(512) ATUS_CASE(1024) ATUS_CASE(2048)
#undef ATUS_CASE
    default: break;
  }
#undef ATUS_K
  return hipErrorInvalidValue;
}

// ------------------------------------------------ resident 1D blocks

constexpr int BCOMP_MOST = 512;  // threads per workgroup: 256 registers each

// The steps whose points cost a few hundred operations at most: one CU holds
// a run, and the three-state and two-species Bragg steps take longer there
// than a pass of their own over the device and its launches do (raman,
// three states, 1024 points: 36 us per step against 19; bragg_ds, 2048
// points: 27 against 15).
#define ATUS_BLOCK_KINDS(X) \
  X(V_NL, 1) X(V_NL_IF, 1) X(V_NL, 2) X(V_NL_IF, 2) X(V_BRAGG, 2) X(V_NL_IF2, 2) X(V_NL, 3) X(V_NL_IF, 3) \
  X(V_NL, 4) X(V_NL_IF, 4) X(V_NL_IF2, 4)

template <int N, int VK, int NC, bool BATCH>
static hipError_t bcomp_go(double2* psi, long long cs, long long runs, const double2* tw, const BlockPhases& ph,
                           const VArgs& va, const BlockSteps& st, double dx0, const Limits& lim, hipStream_t s) {
  constexpr int RM = comp_rm(N, NC, BCOMP_MOST);
  if constexpr (RM == 0 || (NC > 1 && N > 2048)) {
    return hipErrorInvalidValue;
  } else {
    constexpr int T1 = NC * Plan<N, RM>::P;  // threads of one run
    constexpr int LB = T1 <= 256 ? 256 : 512;
    Limits l1 = lim;
    if (!BATCH) l1.threads = 64;  // one run: one pencil
    PassCfg c = comp_cfg(N, RM, NC, runs, l1, LB, block_tw_in_lds<N, NC>());
    if (c.block.x == 0 || c.grid.x == 0) return hipErrorInvalidConfiguration;
    static bool ok = false;
    hipError_t e = allow_lds(k_bcomp<N, RM, VK, NC, BATCH, LB>, c.lds, ok);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_bcomp<N, RM, VK, NC, BATCH, LB>), c.grid, c.block, c.lds, s, psi, cs, c.g, tw, ph, va, st,
                       dx0);
    return hipGetLastError();
  }
}

bool bcomp_ok(int N, int vk, int nc) {
  if ((nc > 1 && N > 2048) || comp_rm(N, nc, BCOMP_MOST) == 0) return false;
#define ATUS_K(V, C) \
  if (vk == V && nc == C) return true;
  ATUS_BLOCK_KINDS(ATUS_K)
#undef ATUS_K
  return false;
}

hipError_t launch_bcomp(int N, int vk, int nc, bool batch, double2* psi, long long comp_stride, long long runs,
                        const double2* tw, const BlockPhases& ph, const VArgs& va, const BlockSteps& st, double dx0,
                        const Limits& lim, hipStream_t s) {
  switch (N) {
#define ATUS_K(V, C) \
  if (!batch && vk == V && nc == C) return bcomp_go<ATUS_N, V, C, false>(psi, comp_stride, runs, tw, ph, va, st, dx0, lim, s);
#define ATUS_CASE(n)                                                                                               \
  case n: {                                                                                                        \
    constexpr int ATUS_N = n;                                                                                      \
    if (batch && nc == 2 && vk == V_BRAGG)                                                                         \
      return bcomp_go<n, V_BRAGG, 2, true>(psi, comp_stride, runs, tw, ph, va, st, dx0, lim, s);                   \
    if (batch && nc == 2 && vk == V_NL_IF)                                                                         \
      return bcomp_go<n, V_NL_IF, 2, true>(psi, comp_stride, runs, tw, ph, va, st, dx0, lim, s);                   \
    ATUS_BLOCK_KINDS(ATUS_K) break;                                                                                 \
  }
    ATUS_CASE(2) ATUS_CASE(4) ATUS_CASE(8) ATUS_CASE(16) ATUS_CASE(32) ATUS_CASE(64) ATUS_CASE(128)
    ATUS_CASE(256) ATUS_CASE(512) ATUS_CASE(1024) ATUS_CASE(2048) ATUS_CASE(4096)
#undef ATUS_CASE
#undef ATUS_K
    default: break;
  }
  return hipErrorInvalidValue;
}

}  // namespace atus
