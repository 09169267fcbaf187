// What the kernels of one wavefront per workgroup share: loads at uniform
// addresses through the scalar cache, the order of LDS accesses.
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

// Orders the LDS accesses of the workgroup's one wavefront: they execute in
// program order, so the compiler's order is all it takes
__device__ __forceinline__ void lds_order()
{
   __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
   __builtin_amdgcn_wave_barrier();
}

// A pointer to device memory that was itself loaded from memory: without
// this the compiler takes it for one that may point to LDS and emits flat
// accesses, which every later wait for LDS waits for too
template <class T>
__device__ __forceinline__ T *in_global(T *p)
{
   return (T *)(__attribute__((address_space(1))) T *)(uintptr_t)p;
}

// Workgroups go round the eight XCDs, each with its own L2, and the items of a
// set quartet read the same blocks: runs of RUN items to one XCD
template <uint32_t RUN>
__device__ __forceinline__ uint32_t xcd_run(uint32_t w, uint32_t n)
{
   constexpr uint32_t XCDS = 8;
   if (w >= n / (RUN * XCDS) * (RUN * XCDS)) return w;
   const uint32_t x = w % XCDS, k = w / XCDS;
   return (k / RUN * XCDS + x) * RUN + k % RUN;
}

// chunk `id` of a launch, with the execution's buffers
__device__ __forceinline__ BatchDev load_batch(const BatchDev *batches, uint32_t id, const RunDev &run)
{
   BatchDev b = load_uniform(batches + id);
   b.tp = in_global(b.tp);
   b.items = in_global(b.items);
   b.segs = in_global(b.segs);
   b.rorder = in_global(b.rorder);
   b.rows = in_global(b.rows);
   b.groups = in_global(b.groups);
   b.prm_row = in_global(b.prm_row);
   b.prm_ip = in_global(b.prm_ip);
   b.ksg = in_global(b.ksg);
   b.kss = in_global(b.kss);
   b.ksx = in_global(b.ksx);
   b.gmag = in_global(b.gmag);
   b.gflag = in_global(b.gflag);
   b.data = in_global(run.data);
   b.ac0 = in_global(run.work + b.ac_off);
   b.eco = in_global(run.work + b.eco_off);
   b.stats = in_global(run.stats);
   b.force_fix = run.force_fix;
   b.id = id;
   if (run.mixed != 1) b.gmag = nullptr;
   if (run.mixed != 2) b.gflag = nullptr;
   return b;
}

}  // namespace gint
