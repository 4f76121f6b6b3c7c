// k_block.hip -- whole blocks of 1D runs of two components and 4096 points in
// one launch (k_block1d).
#include "launch.hpp"

namespace atus {

template <int N, int RM, int VK, int NC, bool BATCH>
static hipError_t block_go(double2* psi, long long cs, long long runs, const double2* tw, const double2* eh,
                           const double2* ef, const VArgs& va, const double* t1tab, const double* Ftab, double dx0,
                           int Nk, const Limits& max_lds, hipStream_t s) {
  // pencils of more than 256 threads (4096 points at 8 values per thread)
  // take workgroups of 512
  constexpr int LB = Plan<N, RM>::P > 256 ? 512 : 256;
  // a single run: one pencil per workgroup; a batch: as many pencils as
  // the workgroup holds
  const int max_threads = BATCH ? LB : threads_per_pencil(N, RM);
  PassCfg c = make_pass_cfg(N, RM, 1, runs, 1, max_lds, 3, max_threads);
  // above 1024 points the twiddle table alone is staged in LDS
  if constexpr (!tables_in_lds<N>()) c.lds += (size_t)N * sizeof(double2);
  if (c.block.x == 0 || c.block.x > LB || c.grid.x == 0 || c.lds > max_lds.lds) return hipErrorInvalidConfiguration;
  static bool ok = false;
  hipError_t e = allow_lds(k_block1d<N, RM, VK, NC, BATCH, LB>, c.lds, ok);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_block1d<N, RM, VK, NC, BATCH, LB>), c.grid, c.block, c.lds, s, psi, cs, c.g, tw, eh, ef, va,
                     t1tab, Ftab, dx0, Nk);
  return hipGetLastError();
}

// two components of 4096 points: a workgroup with a thread group per
// component would need 1024 threads and spill (a batch of 77 runs: 24 us per
// step against 11); everything else runs as launch_bcomp
bool block1d_ok(int N, int vk, int nc) {
  return N == 4096 && nc == 2 && (vk == V_NL || vk == V_NL_IF || vk == V_BRAGG);
}

hipError_t launch_block1d(int vk, bool batch, double2* psi, long long cs, long long runs, const double2* tw,
                          const double2* eh, const double2* ef, const VArgs& va, const double* t1tab,
                          const double* Ftab, double dx0, int Nk, const Limits& lim, hipStream_t s) {
  // 8 values per thread: the pencil gets the most threads to hide latency with
  constexpr int N = 4096, RM = 8;
  if (vk == V_BRAGG)
    return batch ? block_go<N, RM, V_BRAGG, 2, true>(psi, cs, runs, tw, eh, ef, va, t1tab, Ftab, dx0, Nk, lim, s)
                 : block_go<N, RM, V_BRAGG, 2, false>(psi, cs, 1, tw, eh, ef, va, t1tab, Ftab, dx0, Nk, lim, s);
  if (vk == V_NL_IF)
    return batch ? block_go<N, RM, V_NL_IF, 2, true>(psi, cs, runs, tw, eh, ef, va, t1tab, Ftab, dx0, Nk, lim, s)
                 : block_go<N, RM, V_NL_IF, 2, false>(psi, cs, 1, tw, eh, ef, va, t1tab, Ftab, dx0, Nk, lim, s);
  if (vk == V_NL && !batch)
    return block_go<N, RM, V_NL, 2, false>(psi, cs, 1, tw, eh, ef, va, t1tab, Ftab, dx0, Nk, lim, s);
  return hipErrorInvalidValue;
}

}  // namespace atus
