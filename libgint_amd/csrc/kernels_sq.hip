// Launch of k_sq (kernels_sq.hpp).
#include <algorithm>

#include "kernels_sq.hpp"

namespace gint {

#define GINT_SQ_DECL(lm)                                                                                            \
   template <>                                                                                                      \
   int launch_sq_lm<lm>(const BatchDev *, const SqRef *, int, uint32_t, unsigned, size_t, const DevTables &,        \
                        const RunDev &, const KTargets &, void *);
GINT_SQ_DECL(1) GINT_SQ_DECL(2) GINT_SQ_DECL(3) GINT_SQ_DECL(4)
#undef GINT_SQ_DECL

int launch_sq(const BatchDev *batches, const SqRef *refs, int nref, uint32_t items, int lm, size_t lds,
              const DevTables &t, const RunDev &run, const KTargets &kt, void *stream)
{
   if (nref > MAX_LAUNCH_CHUNKS) return -4;
   if (lds > 64 * 1024) return -3;
   // one item per workgroup (a loop over items would keep every argument
   // live); a launch takes at most 2^24 of them (2^30 threads)
   for (uint32_t i0 = 0; i0 < items;) {
      const unsigned grid = std::min(items - i0, 1u << 24);
      int rc;
      switch (lm) {
         case 1: rc = launch_sq_lm<1>(batches, refs, nref, i0, grid, lds, t, run, kt, stream); break;
         case 2: rc = launch_sq_lm<2>(batches, refs, nref, i0, grid, lds, t, run, kt, stream); break;
         case 3: rc = launch_sq_lm<3>(batches, refs, nref, i0, grid, lds, t, run, kt, stream); break;
         default: rc = launch_sq_lm<4>(batches, refs, nref, i0, grid, lds, t, run, kt, stream); break;
      }
      if (rc) return rc;
      i0 += grid;
   }
   return 0;
}

}  // namespace gint
