// k_marg.hip -- densities along one axis (k_marginal).
#include "marg.hpp"

namespace atus {

template <int N, bool CONTIG, bool PHASE>
static hipError_t marg_go(const double2* psi, long long inner, long long outer, const double2* tw, double2* part,
                          double2* out, double* phase, unsigned* nblocks, const Limits& lim, hipStream_t s) {
  constexpr int RM = (N > 8 && N / 8 <= 256) ? 8 : 16;
  PassCfg c = make_pass_cfg(N, RM, inner, outer, 1, lim);
  if (c.block.x == 0 || c.block.x > 256 || c.grid.x == 0) return hipErrorInvalidConfiguration;
  // two workgroups per CU: more would only write more partial sums
  const unsigned nb = c.grid.x < 2u * CU_COUNT ? c.grid.x : 2u * CU_COUNT;
  *nblocks = nb;
  if (!part) return hipSuccess;
  static bool ok = false;
  hipError_t e = allow_lds(k_marginal<N, RM, CONTIG, PHASE>, c.lds, ok);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_marginal<N, RM, CONTIG, PHASE>), dim3(nb), c.block, c.lds, s, psi, c.g, tw, part, phase);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_marginal_sum, dim3((N + 15) / 16), dim3(256), 0, s, part, (int)nb, N, out);
  return hipGetLastError();
}

hipError_t launch_marginal(int N, const double2* psi, long long inner, long long outer, const double2* tw,
                           double2* part, double2* out, double* phase, unsigned* nblocks, const Limits& lim,
                           hipStream_t s) {
  if (phase && inner != 1) return hipErrorInvalidValue;
  switch (N) {
#define ATUS_CASE(n)                                                                                        \
  case n:                                                                                                   \
    if (inner != 1) return marg_go<n, false, false>(psi, inner, outer, tw, part, out, phase, nblocks, lim, s); \
    return phase ? marg_go<n, true, true>(psi, inner, outer, tw, part, out, phase, nblocks, lim, s)         \
                 : marg_go<n, true, false>(psi, inner, outer, tw, part, out, phase, nblocks, lim, s);
    ATUS_CASE(2) ATUS_CASE(4) ATUS_CASE(8) ATUS_CASE(16) ATUS_CASE(32) ATUS_CASE(64) ATUS_CASE(128)
    ATUS_CASE(256) ATUS_CASE(512) ATUS_CASE(1024) ATUS_CASE(2048) ATUS_CASE(4096)
#undef ATUS_CASE
    default: return hipErrorInvalidValue;
  }
}

}  // namespace atus
