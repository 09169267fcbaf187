// Launch of k_sq (kernels_sq.hpp).
#include <algorithm>

#include "kernels_sq.hpp"

namespace gint {

template <>
int launch_sq_lm<1>(const BatchDev &, const DevTables &, const KTargets &, const SqArgs &, unsigned, size_t, void *);
template <>
int launch_sq_lm<2>(const BatchDev &, const DevTables &, const KTargets &, const SqArgs &, unsigned, size_t, void *);
template <>
int launch_sq_lm<3>(const BatchDev &, const DevTables &, const KTargets &, const SqArgs &, unsigned, size_t, void *);

int launch_sq(const TypePlan &tp, int max_np, const BatchDev &b, const DevTables &t, const KTargets &kt,
              const SqPlan &sp, void *stream)
{
   if (b.g1 <= b.g0 || sp.items.empty()) return 0;
   const char *dev = (const char *)sp.dev;
   SqArgs y;
   y.items = (const SqItem *)(dev + sp.off[0]);
   y.tiles = (const SqTile *)(dev + sp.off[1]);
   y.sps = (const SqSp *)(dev + sp.off[2]);
   y.rows = (const uint16_t *)(dev + sp.off[3]);
   y.rcs = (const uint32_t *)(dev + sp.off[4]);
   y.fns = (const uint32_t *)(dev + sp.off[5]);
   y.nitem = (int)sp.items.size();
   int ncon = 0;
   for (int x = 0; x < 4; x++) {
      y.ncon[x] = 0;
      for (int s = 0; s < tp.nsh[x]; s++) y.ncon[x] += tp.nl[x][s];
      ncon += y.ncon[x];
   }
   y.o_co = sp.lds_bytes / 8;
   const size_t lds = (size_t)sp.lds_bytes + 8 * (size_t)(ncon * max_np);
   if (lds > 64 * 1024) return -3;
   // one item per workgroup (a loop over items would keep every argument
   // live); a launch takes at most 2^24 of them (2^30 threads)
   const uint32_t step = std::max(1u, (1u << 24) / (uint32_t)y.nitem);
   BatchDev c = b;
   for (uint32_t g0 = b.g0; g0 < b.g1; g0 += std::min(step, b.g1 - g0)) {
      c.g0 = g0;
      c.g1 = g0 + std::min(step, b.g1 - g0);
      const unsigned grid = (c.g1 - c.g0) * (unsigned)y.nitem;
      int rc;
      switch (sp.lm) {
         case 1: rc = launch_sq_lm<1>(c, t, kt, y, grid, lds, stream); break;
         case 2: rc = launch_sq_lm<2>(c, t, kt, y, grid, lds, stream); break;
         default: rc = launch_sq_lm<3>(c, t, kt, y, grid, lds, stream); break;
      }
      if (rc) return rc;
   }
   return 0;
}

}  // namespace gint
