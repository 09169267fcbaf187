// One k_sq instantiation (the shell pairs it has code for: has_pair) per
// translation unit (-DGINT_SQ_LM=<1..4>), compiled side by side.
#include "kernels_sq.hpp"

#ifndef GINT_SQ_LM
#error "build with -DGINT_SQ_LM=<1..4>"
#endif

namespace gint {

template <>
int launch_sq_lm<GINT_SQ_LM>(const BatchDev *batches, const SqRef *refs, int nref, uint32_t item0, unsigned grid, size_t lds,
                             const DevTables &t, const RunDev &run, const KTargets &kt, void *stream)
{
   hipLaunchKernelGGL((sq::k_sq<GINT_SQ_LM>), dim3(grid), dim3(64), lds, (hipStream_t)stream, batches, refs, nref, item0, t,
                      run, kt);
   return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace gint
