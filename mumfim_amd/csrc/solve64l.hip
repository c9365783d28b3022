// solve64 with the incidence lists in LDS, in a file of its own so that the
// constants of its exponential stay in registers over the step loop: these
// shapes have registers to spare, and formed anew for every fiber the constants
// cost 3-7% (1024 RVEs of 250 and 500 nodes with energies, 300 steps: linear
// 4.40 and 8.39 against 4.40 and 8.22 ms, half toe law 6.45 and 12.6 against
// 6.16 and 11.8).  The 1024-thread shapes are the other way round: their
// constants spill (1000 nodes: linear 9.8 against 6.5 ms).
#include "solve64_ieee.hpp"

namespace mf {

hipError_t launch_solve64l(const Variant &v, const SolveArgs &a, int n_blocks, size_t lds,
                           hipStream_t s) {
#define MF_VARIANT_LAUNCH(P, B, N, F)                                        \
  if constexpr (P == MF_PREC_FP64 && ((F) & kEllInLds))                      \
    if (v.block == B && v.npt == N && (v.flags & ~kEnergy) == F) {           \
      auto k = (v.flags & kEnergy) ? kern::solve64<B, N, F, true>            \
                                   : kern::solve64<B, N, F, false>;          \
      if (lds > 64 * 1024)                                                   \
        (void)hipFuncSetAttribute((const void *)k,                           \
                                  hipFuncAttributeMaxDynamicSharedMemorySize, \
                                  (int)kMaxLds);                             \
      hipLaunchKernelGGL(k, dim3(n_blocks), dim3(B), lds, s, a);             \
      return hipGetLastError();                                              \
    }
  MF_VARIANT_LIST(MF_VARIANT_LAUNCH)
#undef MF_VARIANT_LAUNCH
  return hipErrorInvalidValue;
}

}  // namespace mf
