// The host loop of a trip-scheduled call on the CPU: kernels run serially as in emu.cpp,
// while launches, synchronisations and events are counted the way a stream orders them,
// so that a test can ask which kernels the host has not waited for when the call returns.
// One mechanism, chosen on the compiler's command line (PELE_TU_MECH and its companions).
#define PELE_WAVES_PER_EU(n)
#include <cstring>
#include <vector>

#include "hip/hip_runtime.h"

namespace host {
// kernels launched, and how many of them the host knows to have finished
static long launched = 0, waited = 0, looks = 0;
static long recorded = 0;   // launches before the last event record (one event is used)
inline hipError_t stream_sync(hipStream_t) {
  waited = launched;
  return hipSuccess;
}
inline hipError_t record(hipEvent_t, hipStream_t) {
  recorded = launched;
  return hipSuccess;
}
inline hipError_t event_sync(hipEvent_t) {
  if (recorded > waited) waited = recorded;
  return hipSuccess;
}
inline hipError_t copy(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t st) {
  if (k == hipMemcpyDeviceToHost) ++looks;
  return hipMemcpyAsync(d, s, n, k, st);
}
}  // namespace host

#undef hipLaunchKernelGGL
#define hipLaunchKernelGGL(kernel, grid, block, shmem, stream, ...)             \
  do {                                                                         \
    const dim3 g_ = (grid), b_ = (block);                                      \
    ++host::launched;                                                          \
    blockDim.x = b_.x;                                                         \
    gridDim.x = g_.x;                                                          \
    for (unsigned bx_ = 0; bx_ < g_.x; ++bx_)                                  \
      for (unsigned tx_ = 0; tx_ < b_.x; ++tx_) {                              \
        blockIdx.x = bx_;                                                      \
        threadIdx.x = tx_;                                                     \
        kernel(__VA_ARGS__);                                                   \
      }                                                                        \
  } while (0)
#define hipStreamSynchronize host::stream_sync
#define hipEventRecord host::record
#define hipEventSynchronize host::event_sync
#define hipMemcpyAsync host::copy

#include "../../pelelm_amd/csrc/reactor_bdf.hip"

thread_local Idx3 threadIdx, blockIdx, blockDim, gridDim;

using namespace pelelm;

// One react call on flat cell-fastest arrays.  ahead = 1 gives the call the pinned counts
// and the event with which it issues a trip's evaluation before it waits; profile = 1 has
// its kernels timed, for which trips come one by one and each evaluation after the wait; out: kernels
// launched, kernels not waited for at the return, looks at the device's counts, trips.
extern "C" int host_react(long ncell, double* rY, double* T, double* rE, double* FC, double dt, double rtol,
                          double atol, int compact, int gmres, int ahead, int profile, long max_trips, unsigned long long* counters,
                          long* out) {
  const MechTable* t = PELE_TU_MECH_FN();
  const int N = t->nspec;
  ReactArgs a{};
  a.rY.p = rY; a.rY.ns = ncell;
  a.T.p = T; a.T.ns = ncell;
  a.rE.p = rE; a.rE.ns = ncell;
  a.FC.p = FC; a.FC.ns = ncell;
  a.nx = (int)ncell; a.ny = 1; a.ncell = ncell;
  a.dt = dt; a.rtol = rtol;
  for (int i = 0; i <= N; ++i) a.atol[i] = atol;
  a.qmax = 4; a.mxstep = 20000;
  const size_t n64 = (size_t)((ncell + 63) / 64) * 64;
  std::vector<double> ws(n64 * t->ws_slots), mat(n64 * t->mat_stride);
  std::vector<int> iws(n64 * t->iws_slots + 1), lists(6 * n64);
  std::memset(ws.data(), 0xFF, ws.size() * sizeof(double));
  std::memset(mat.data(), 0xFF, mat.size() * sizeof(double));
  unsigned int counts[8] = {0}, pinned[8];
  a.ws = ws.data(); a.iws = iws.data(); a.mat = mat.data();
  for (int i = 0; i < 2; ++i) {
    a.list[i] = lists.data() + i * n64;
    a.slist[i] = lists.data() + (2 + i) * n64;
  }
  a.plist = lists.data() + 4 * n64;
  a.nlist = lists.data() + 5 * n64;
  a.counts = counts;
  a.counters = counters;
  a.compact = compact;
  a.gmres = gmres;
  a.gmres_maxl = 5;
  a.lu_lane = 1;
  a.lu_mode = LU_FP64;
  a.ir_tol = 1e-4;
  TripPlan plan;
  int event = 0;
  if (ahead) {
    plan.host_counts = pinned;
    plan.counted = &event;
  }
  host::launched = host::waited = host::looks = host::recorded = 0;
  KernelProf prof{};
  const int rc = (int)t->run_react(a, nullptr, max_trips, &out[3], profile ? &prof : nullptr, nullptr, plan);
  out[0] = host::launched;
  out[1] = host::launched - host::waited;
  out[2] = host::looks;
  return rc;
}
