// Loads at uniform addresses through the scalar cache, for the kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "device.hpp"

namespace gint {

// A record at a uniform address, through the scalar cache: nothing that a
// kernel of the K-build reads this way is written by one (plans, records,
// tables and basis data), which the compiler cannot see behind the stores
template <class T>
__device__ __forceinline__ T load_uniform(const T *p)
{
   static_assert(sizeof(T) % 4 == 0, "whole words");
   typedef const __attribute__((address_space(4))) uint32_t *word_ptr;
   const word_ptr q = (word_ptr)(uintptr_t)p;
   union {
      uint32_t w[sizeof(T) / 4];
      T v;
   } u;
#pragma unroll
   for (unsigned i = 0; i < sizeof(T) / 4; i++) u.w[i] = q[i];
   return u.v;
}

// chunk `id` of a launch, with the execution's buffers
__device__ __forceinline__ BatchDev load_batch(const BatchDev *batches, uint32_t id, const RunDev &run)
{
   BatchDev b = load_uniform(batches + id);
   b.data = run.data;
   b.ac0 = run.work + b.ac_off;
   b.eco = run.work + b.eco_off;
   b.stats = run.stats;
   b.fix = run.fix;
   b.fix_count = run.fix_count;
   b.fix_ws = run.fix_ws;
   b.fix_cap = run.fix_cap;
   b.fix_stride = run.fix_stride;
   b.force_fix = run.force_fix;
   b.id = id;
   if (run.mixed != 1) b.gmag = nullptr;
   if (run.mixed != 2) b.gflag = nullptr;
   return b;
}

}  // namespace gint
