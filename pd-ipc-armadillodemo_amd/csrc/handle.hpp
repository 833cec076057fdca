// The library handle shared by the step driver (pdipc_api.hip) and the adjoint
// (adjoint.hip), plus the host helpers both use.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>
#include <vector>

#include "../../include/pdipc.h"
#include "device.hpp"
#include "host_setup.hpp"

namespace pdipc {

int fail(int code, const std::string& msg);

#define HIPCHK(expr)                                                                          \
  do {                                                                                        \
    hipError_t e_ = (expr);                                                                   \
    if (e_ != hipSuccess) return ::pdipc::fail(PDIPC_E_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

struct AdjointState;                 // adjoint.hip
void adjoint_free(AdjointState* a);  // releases its device memory

}  // namespace pdipc

using pdipc::fail;

struct pdipc_handle;
namespace pdipc {
void noalloc_release(pdipc_handle* h);  // noalloc.hip: gives the slot of its minima back
}

struct pdipc_handle {
  using HostSetup = pdipc::HostSetup;
  using SellLayout = pdipc::SellLayout;
  using DeviceMesh = pdipc::DeviceMesh;
  using ModelInput = pdipc::ModelInput;
  pdipc_params prm;
  std::vector<ModelInput> sims, statics;
  bool hostReady = false, deviceReady = false;
  HostSetup hs;
  SellLayout sell;
  DeviceMesh m;
  hipStream_t stream = nullptr;
  int device = 0;  // the HIP device current at pdipc_init
  double* toiMinima = nullptr;  // where pdipc_toi_noalloc keeps its workgroup minima,
  int toiSlot = -1;             // and the slot of the device's array it is (-1: the handle's own buffer)
  // local/global loop captured once per (tile solves, collision flag, precision) and replayed
  hipGraphExec_t lgGraph[2][2][2] = {};
  int tileAborts = 0;  // outer iterations repeated with the streamed sweeps,
  int tileStreak = 0;  // of them the last in a row less than a minute apart,
  double tileLastAbort = 0.0, tileRest = 0.0;  // when the last one was, and until when no tile solve is tried
  std::vector<void*> allocs;
  // host mirrors
  void* scalHost = nullptr;  // pinned, after `stage`: residual, toiBits, counters[12], the tile solves' abort flag
  void* scalDev = nullptr;
  double* stage = nullptr;   // pinned: 3 * ld doubles, arrays of points on their way in or out
  pdipc_counters cnt;
  int lastRecs = 0, lastPairs = 0;
  double* trackToi = nullptr;  // per-record TOIs when track_toi_argmin is on
  int trackCap = 0;

  template <class T>
  int alloc(T** p, size_t n) {
    size_t bytes = std::max<size_t>(n, 1) * sizeof(T);
    hipError_t e = hipMalloc((void**)p, bytes);
    if (e != hipSuccess) return fail(PDIPC_E_HIP, std::string("hipMalloc: ") + hipGetErrorString(e));
    allocs.push_back(*p);
    return PDIPC_OK;
  }
  // Copies and waits on the handle's own stream: the legacy stream must not be
  // used while another thread's handle captures its graphs.
  hipError_t copy(void* dst, const void* src, size_t bytes, hipMemcpyKind kind) {
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, stream);
    return e != hipSuccess ? e : hipStreamSynchronize(stream);
  }
  template <class T>
  int upload(T** p, const std::vector<T>& v) {
    int rc = alloc(p, v.size());
    if (rc) return rc;
    if (!v.empty()) HIPCHK(copy(*p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return PDIPC_OK;
  }
  void release(void* p) {
    if (!p) return;
    auto it = std::find(allocs.begin(), allocs.end(), p);
    if (it != allocs.end()) allocs.erase(it);
    (void)hipFree(p);
  }
  pdipc::AdjointState* adj = nullptr;
  ~pdipc_handle() {
    if (stream) (void)hipStreamSynchronize(stream);
    drop_graphs();  // the executable graphs go before the buffers their nodes point to
    delete m.timer;
    pdipc::adjoint_free(adj);
    for (void* p : allocs) (void)hipFree(p);
    pdipc::noalloc_release(this);  // (the frees have waited for the device)
    if (stage) (void)hipHostFree(stage);
    if (stream) (void)hipStreamDestroy(stream);
  }
  void drop_graphs() {
    for (auto& tiles : lgGraph)
      for (auto& row : tiles)
        for (auto& g : row)
          if (g) {
            (void)hipGraphExecDestroy(g);
            g = nullptr;
          }
  }
  double* hResidual() { return (double*)scalHost; }
  unsigned long long* hToi() { return (unsigned long long*)((char*)scalHost + 8); }
  int* hCounters() { return (int*)((char*)scalHost + 16); }
  int hTileAbort() { return *(int*)((char*)scalHost + 64); }
};


namespace pdipc {
int put_soa(pdipc_handle* h, double* dst, const double* aos, int npts);
int put_soa_prefix(pdipc_handle* h, double* dst, const double* aos, int npts);
int get_soa(pdipc_handle* h, const double* src, double* aos, int npts);
int check_launch(pdipc_handle* h);
int read_scalars(pdipc_handle* h);
int broad_phase(pdipc_handle* h, const double* x, const double* dx);
int collision(pdipc_handle* h);
int require_device(pdipc_handle* h);
int advance(pdipc_handle* h);
// The tile solves wait for each other, so only one handle per device launches
// them at a time: a call that runs solves holds the device's turn for its
// duration, or, when another thread's handle has it, runs the streamed sweeps
// (the same results bit for bit).
class TileTurn {
 public:
  explicit TileTurn(pdipc_handle* h);
  ~TileTurn();
  void renew();  // before each step of the call: tile solves may run, or again
  TileTurn(const TileTurn&) = delete;
  TileTurn& operator=(const TileTurn&) = delete;

 private:
  pdipc_handle* h_;
  bool held_ = false;
};
// returned by read_scalars (and what calls it) when a tile solve gave up
// waiting; tile_recover clears the flag, switches the handle to the streamed
// sweeps until the turn is renewed and restores X as the outer iteration
// found it
constexpr int kTileAborted = 1000;
int tile_recover(pdipc_handle* h, int outer);
void tile_gave_up(pdipc_handle* h);  // counts it, and may have the handle rest from tile solves
int adjoint_refresh_values(pdipc_handle* h);  // adjoint.hip: after a stiffness change
int noalloc_setup(pdipc_handle* h);            // noalloc.hip: with the handle's device current
}  // namespace pdipc
