// The host engine on the CPU: a HIP runtime over host memory and launchers
// that do no work, so that the tests can drive queues, plans and the request
// loop without a GPU.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <utility>
#include <vector>

#include "device.hpp"

namespace {
template <class T>
hipError_t handle(T *h)
{
   *h = (T)std::malloc(8);
   return hipSuccess;
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t n)
{
   *p = std::calloc(n ? n : 1, 1);
   return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p)
{
   std::free(p);
   return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
   std::memcpy(d, s, n);
   return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemset(void *d, int v, size_t n)
{
   std::memset(d, v, n);
   return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t s) { return hipFree(s); }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return handle(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return hipFree(e); }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
   *ms = 0.f;
   return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return handle(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) { return handle(e); }
hipError_t hipGraphDestroy(hipGraph_t g) { return hipFree(g); }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { return hipFree(e); }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stub"; }
}

namespace gint {

void *noalloc_scratch()
{
   static void *p = std::calloc(NOALLOC_BYTES, 1);
   return p;
}
int launch_zero_u32(uint32_t *p, int n, void *)
{
   std::memset(p, 0, 4 * (size_t)n);
   return 0;
}
void launch_zero_f64(double *p, size_t n, void *) { std::memset(p, 0, 8 * n); }
int launch_fm_r(const BatchDev *, const WorkRef *, int, uint32_t, int, size_t, const DevTables &, const RunDev &, void *) { return 0; }
// the fix-up entries of the last launch's chunks
static std::vector<std::pair<uint32_t, uint32_t>> g_fix;
int launch_fixup(const BatchDev *b, int n, size_t, const DevTables &, const RunDev &, uint32_t, void *)
{
   g_fix.clear();
   for (int i = 0; i < n; i++) g_fix.emplace_back(b[i].fix_at, b[i].fix_cap);
   return 0;
}
int launch_sq(const BatchDev *, const SqRef *, int, uint32_t, int, size_t, const DevTables &, const RunDev &, const KTargets &, void *)
{
   return 0;
}
int launch_eco(const BatchDev *, const RunDev &, uint32_t, const EcoArgs &, void *) { return 0; }
int launch_absmax(const double *, size_t, unsigned long long *, bool, void *) { return 0; }
int launch_mixed_flags(const BatchDev *, const RunDev &, uint32_t, const unsigned long long *, double, unsigned long long *, void *)
{
   return 0;
}
int launch_pack_c0(const double *, int, int, double *, void *) { return 0; }
int device_math_selftest(const double *, const double *, int, double *) { return -1; }
int mfma_selftest(const double *, const double *, double *, int) { return -1; }
size_t fm_r_lds_bytes(const TypePlan &) { return 1024; }
void fm_layouts(const TypePlan &, FmLayout &main, FmLayout &fix)
{
   main = fix = FmLayout{};
   main.NB = 16;
   fix.NB = 1;
   main.bytes = fix.bytes = 1024;
}

}  // namespace gint

extern "C" {
int stub_fix_chunks() { return (int)gint::g_fix.size(); }
int stub_fix_at(int i) { return (int)gint::g_fix[i].first; }
int stub_fix_cap(int i) { return (int)gint::g_fix[i].second; }
}
