// pdipc_toi_noalloc: the minimum ACCD time of impact over the current
// candidate records (what pdipc_debug_toi returns) for callers that cannot
// allocate device memory -- code under HIP graph capture, tight serving loops.
// Positions and the result stay on the device, the work is only enqueued, and
// the per-workgroup minima live in `scratch`, a file-scope device array each
// GPU holds for the life of the process: a handle has a slot of it from
// pdipc_init to pdipc_destroy (a call writes at most 2,048 minima), or, while
// 32 others have them all, a buffer of its own allocated at pdipc_init.  The
// array's device address comes from hipGetSymbolAddress once per device
// (pdipc_init, with the handle's device current); host code passes that
// address, never the array's name.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <mutex>
#include <string>

#include "handle.hpp"

namespace pdipc {

namespace {

constexpr int kMaxRecs = 1 << 24;      // candidate records a call takes
constexpr int kSlots = 32;             // handles that have a part of `scratch` at a time
constexpr int kMaxDevices = 64;
constexpr int kReduceThreads = 1024;

static_assert(kSlots == 32, "one bit of g_taken each");
static __device__ __align__(256) double scratch[kSlots * kMaxToiBlocks];

std::mutex g_mu;
double* g_scratch[kMaxDevices] = {};  // device address of `scratch`, per device
uint32_t g_taken[kMaxDevices] = {};   // bit per slot: some handle has it

// one workgroup: min over the n block minima, then the reference's safety
// scale (getImpactOfTimeHost, PdIpcGpuFunc.cu:2698-2699): t < 1 -> t * scale
__global__ void __launch_bounds__(kReduceThreads) k_toi_reduce(const double* __restrict__ blockMin, int n,
                                                               double scale, double* __restrict__ out) {
  __shared__ double part[kReduceThreads];
  double m = 1.0;
  for (int i = threadIdx.x; i < n; i += kReduceThreads) {
    double v = blockMin[i];
    m = v < m ? v : m;
  }
  part[threadIdx.x] = m;
  __syncthreads();
  for (int o = kReduceThreads / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      double v = part[threadIdx.x + o];
      part[threadIdx.x] = v < part[threadIdx.x] ? v : part[threadIdx.x];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = part[0] < 1.0 ? part[0] * scale : 1.0;
}

}  // namespace

// With the handle's device current: its place for the minima.  This device's
// copy of `scratch` is looked up once.
int noalloc_setup(pdipc_handle* h) {
  const int device = h->device;
  if (device < 0 || device >= kMaxDevices) return fail(PDIPC_E_ARG, "device ordinal out of range");
  if (h->toiMinima) return PDIPC_OK;
  std::lock_guard<std::mutex> lock(g_mu);
  if (!g_scratch[device]) {
    void* p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(PDIPC_E_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    g_scratch[device] = (double*)p;
  }
  if (g_taken[device] == ~0u) return h->alloc(&h->toiMinima, kMaxToiBlocks);
  h->toiSlot = __builtin_ctz(~g_taken[device]);
  g_taken[device] |= 1u << h->toiSlot;
  h->toiMinima = g_scratch[device] + (size_t)h->toiSlot * kMaxToiBlocks;
  return PDIPC_OK;
}

void noalloc_release(pdipc_handle* h) {
  if (h->toiSlot < 0) return;
  std::lock_guard<std::mutex> lock(g_mu);
  g_taken[h->device] &= ~(1u << h->toiSlot);
  h->toiSlot = -1;
}

}  // namespace pdipc

using namespace pdipc;

int pdipc_toi_noalloc(pdipc_handle* h, const double* x0, const double* x1, double* toi, void* stream) {
  int rc = require_device(h);
  if (rc) return rc;
  if (!x0 || !x1 || !toi) return fail(PDIPC_E_ARG, "null argument");
  const int nRecs = h->lastRecs;
  if (nRecs > kMaxRecs)
    return fail(PDIPC_E_CAPACITY, "pdipc_toi_noalloc: " + std::to_string(nRecs) +
                                      " candidate records exceed its limit of 16777216 (use pdipc_debug_toi)");
  hipStream_t s = stream ? (hipStream_t)stream : h->stream;
  const pdipc_params& p = h->prm;
  const int minima = launch_ccd_blockmin(h->m, nRecs, x0, x1, p.ccd_filter, p.ccd_iters, p.ccd_step, p.ccd_gap,
                                         p.touch_policy, h->toiMinima, s);
  hipLaunchKernelGGL(k_toi_reduce, dim3(1), dim3(kReduceThreads), 0, s, h->toiMinima, minima, p.toi_scale, toi);
  return check_launch(h);
}
