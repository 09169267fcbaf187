// The k_sq instantiation for angular momenta up to GINT_SQ_LM: one
// translation unit each (-DGINT_SQ_LM=<1..3>), compiled side by side.
#include "kernels_sq.hpp"

#ifndef GINT_SQ_LM
#error "build with -DGINT_SQ_LM=<1..3>"
#endif

namespace gint {

template <>
int launch_sq_lm<GINT_SQ_LM>(const BatchDev &b, const DevTables &t, const KTargets &kt, const SqArgs &y, unsigned grid,
                             size_t lds, void *stream)
{
   hipLaunchKernelGGL((sq::k_sq<GINT_SQ_LM>), dim3(grid), dim3(64), lds, (hipStream_t)stream, b.tp, t, b, kt, y);
   return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace gint
