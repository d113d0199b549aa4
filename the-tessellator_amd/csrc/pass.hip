// pass.hip -- what a call does before and between its passes: counters
// cleared in one launch, and everything the host must know written to pinned
// host memory in one launch.
#include "launch.h"

namespace tess {

namespace {

__global__ __launch_bounds__(256) void k_pass_begin(PassCounters a) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  constexpr uint32_t kSlotWords = sizeof(SummarySlot) / 4;
  if (a.summary && i < kSummarySlots * kSlotWords) reinterpret_cast<uint32_t*>(a.summary)[i] = 0u;
  if (a.arena && i < 2 * kArenaWords) reinterpret_cast<uint32_t*>(a.arena)[i] = 0u;
  if (i < 3) {
    uint32_t* p = i == 0 ? a.redo : i == 1 ? a.tredo : a.spill;
    if (p) *p = 0u;
  }
}

// One wavefront: lane k holds summary slot k, lane 0 the rest.  Bound by its
// launch and the round trip; a hipMemcpyAsync per word into pageable memory
// took 13 us each, and a call had eight (with the clears and the scans below
// 16,384 counts in one launch each: a diagram of 1,000 points 420 -> 267 us,
// of 10,000 593 -> 448).
__global__ __launch_bounds__(64) void k_pass_report(ReportArgs a, PassReport* __restrict__ out) {
  const int lane = threadIdx.x;
  static_assert(kSummarySlots == 64, "a slot per lane");
  Summary s{};
  if (a.summary) s = a.summary[lane].s;
#pragma unroll
  for (int m = 1; m < 64; m *= 2) {
    s.flops += __shfl_xor(s.flops, m);
    s.incident_cuts += __shfl_xor(s.incident_cuts, m);
    s.degenerate += __shfl_xor(s.degenerate, m);
  }
  if (lane == 0) {
    PassReport r{};
    r.sum = s;
    if (a.redo) r.nredo = *a.redo;
    if (a.tredo) r.ntab = *a.tredo;
    if (a.spill) r.nspill = *a.spill;
    if (a.binned) r.binned = *a.binned;
    if (a.total) r.total = *a.total;
    if (a.extra) r.extra = *a.extra;
    if (a.grid) r.grid = *a.grid;
    *out = r;
  }
}

}  // namespace

hipError_t launch_pass_begin(const PassCounters& a, hipStream_t s) {
  constexpr uint32_t slots = kSummarySlots * sizeof(SummarySlot) / 4, words = slots > 2 * kArenaWords ? slots : 2 * kArenaWords;
  hipLaunchKernelGGL(k_pass_begin, dim3((words + 255) / 256), dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_pass_report(const ReportArgs& a, PassReport* host, hipStream_t s) {
  hipLaunchKernelGGL(k_pass_report, dim3(1), dim3(64), 0, s, a, host);
  return hipGetLastError();
}

}  // namespace tess
