// table.hip -- shell tables (celery.rs:418-679) built on the device: the
// offsets of a grid shape in canonical order, one launch for one or many
// shapes.
#include "launch.h"

namespace tess {

namespace {

constexpr int kTableLanes = 16;  // per offset
constexpr int kTableClasses = kTableDeviceL * kTableDeviceL * kTableDeviceL;

// Members of a class (gaps packed ga | gb << 8 | gc << 16) generated before g.
// Gap 0 of an axis holds o = -1, 0 and 1, the others two offsets each.
__device__ uint32_t class_before(int64_t cpd, uint32_t gaps, uint64_t g) {
  const int ga = gaps & 255, gb = (gaps >> 8) & 255, gc = gaps >> 16;
  uint32_t before = 0;
  for (int a = -1; a <= 1; a += ga ? 2 : 1)
    for (int b = -1; b <= 1; b += gb ? 2 : 1)
      for (int c = -1; c <= 1; c += gc ? 2 : 1) {
        if (!a && !b && !c) continue;  // the centre
        before += shell_generation(cpd, a * (ga + 1), b * (gb + 1), c * (gc + 1)) < g ? 1u : 0u;
      }
  return before;
}

// An offset's place is the number of offsets before it.  Keys depend on the
// gaps |o| - 1 alone, so at L rings there are L^3 of them (1,728 at L = 12,
// of 15,625 offsets): an offset counts the members of the classes with a
// smaller key, and looks into a class only where the keys are equal, for the
// members generated before it.  Sixteen lanes per offset; the classes of equal
// key are noted on the way and looked into afterwards, when all lanes have
// theirs.  Bound by the walk over the classes in LDS.  12 rings: 470 us on a
// host thread (sorting 15,625 entries, upload not counted), 22 us here (40
// with four lanes per offset); 64 tables 450 us.
__global__ __launch_bounds__(256) void k_table(const TableBuild* __restrict__ many, TableBuild one) {
  __shared__ double key[kTableClasses];
  __shared__ uint32_t info[kTableClasses];  // gaps, members << 24
  const TableBuild T = many ? many[blockIdx.y] : one;
  const int L = T.L, w = 2 * L + 1, n = w * w * w, nc = L * L * L;
  const int e = blockIdx.x * (256 / kTableLanes) + threadIdx.x / kTableLanes, part = threadIdx.x % kTableLanes;
  if (blockIdx.x * (256 / kTableLanes) >= n) return;
  for (int c = threadIdx.x; c < nc; c += 256) {
    const int ga = c / (L * L), gb = c / L % L, gc = c % L;
    key[c] = shell_gap_key(ga, gb, gc, T.sx, T.sy, T.sz);
    const int members = (ga ? 2 : 3) * (gb ? 2 : 3) * (gc ? 2 : 3) - (c == 0 ? 1 : 0);  // less the centre
    info[c] = (uint32_t)(ga | gb << 8 | gc << 16 | members << 24);
  }
  __syncthreads();
  const bool live = e < n;
  const int ei = live ? e : 0;
  const int ox = ei / (w * w) - L, oy = ei / w % w - L, oz = ei % w - L;
  const bool centre = !ox && !oy && !oz;
  const double k = shell_key(ox, oy, oz, T.sx, T.sy, T.sz);
  const uint64_t g = shell_generation(T.cpd, ox, oy, oz);
  uint32_t before = 0;
  uint64_t equal = ~0ull;  // up to four classes, 16 bits each
  if (!centre) {
#pragma unroll 4
    for (int c = part; c < nc; c += kTableLanes) {
      const double kc = key[c];
      const uint32_t i = info[c];
      before += kc < k ? i >> 24 : 0u;
      if (kc == k) {
        if (equal >> 48 != 0xffff) before += class_before(T.cpd, info[equal >> 48] & 0xffffff, g);
        equal = equal << 16 | (uint64_t)c;
      }
    }
    while (equal != ~0ull) {
      const uint32_t c = (uint32_t)equal & 0xffff;
      before += class_before(T.cpd, info[c] & 0xffffff, g);
      equal = equal >> 16 | 0xffffull << 48;
    }
  }
#pragma unroll
  for (int m = 1; m < kTableLanes; m *= 2) before += __shfl_xor(before, m);
  if (!centre) before += 1;  // the centre comes first
  const bool kept = T.L == T.cpd - 1 || k < T.kcut;
  if (live && part == 0 && kept && before < (uint32_t)T.len) {
    T.key[before] = k;
    T.off[before] = pack_off(ox, oy, oz);
  }
}

}  // namespace

// Sets of a batch in grid y, whose documented limit is 65,536 on this device:
// batches of more sets take several launches.
constexpr int kTableSets = 32768;

hipError_t launch_table(const TableBuild* many, int count, const TableBuild& one, hipStream_t s) {
  const int w = 2 * one.L + 1;
  const dim3 block(256);
  const unsigned x = (unsigned)((w * w * w * kTableLanes + 255) / 256);
  if (!many) {
    hipLaunchKernelGGL(k_table, dim3(x, 1), block, 0, s, many, one);
    return hipGetLastError();
  }
  for (int at = 0; at < count; at += kTableSets) {
    const int n = count - at < kTableSets ? count - at : kTableSets;
    hipLaunchKernelGGL(k_table, dim3(x, (unsigned)n), block, 0, s, many + at, one);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace tess
