// Launches of the tangent-linear kernels; here one direction on 1024 threads
// with up to two nodes per lane.  Compiled as the other FP32 files are: with the
// flag of solve32tk.hip linear RVEs took 3-5% longer (64 RVEs of 1950 nodes, 200
// steps: 2.36 -> 2.48 ms).
#include "solve32t.hpp"

namespace mf {

// the other shapes
hipError_t launch_solve32tk(const Variant &v, const SolveArgs &a, int n_blocks, size_t lds,
                            hipStream_t s);

hipError_t launch_solve32t(const Variant &v, const SolveArgs &a, int n_blocks, size_t lds,
                           hipStream_t s) {
#define MF_TL_LAUNCH(B, N)                                                   \
  if (v.block == B && v.npt == N && variant_fpl(v.flags) == 0) {             \
    auto k = kern::solve32t<B, N>;                                           \
    if (lds > 64 * 1024)                                                     \
      (void)hipFuncSetAttribute((const void *)k,                             \
                                hipFuncAttributeMaxDynamicSharedMemorySize, \
                                (int)kMaxLds);                               \
    hipLaunchKernelGGL(k, dim3(n_blocks), dim3(B), lds, s, a);               \
    return hipGetLastError();                                                \
  }
  MF_TL_LIST(MF_TL_LAUNCH)
#undef MF_TL_LAUNCH
  return launch_solve32tk(v, a, n_blocks, lds, s);
}

}  // namespace mf
