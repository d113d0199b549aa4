// shuffle.hip -- the sample order of a training epoch on the device.
//
// The order is Fisher and Yates's: for i = n - 1 ... 1 swap p[i] with p[h(i)],
// h(i) = splitmix64 mod (i + 1), p the identity at first.  The swaps need not
// be made one after the other: p[i] is final once i's swap is done, and what
// it got lay in place h(i) then, put there by the last earlier swap that
// wrote to h(i), k = min { k > i : h(k) = h(i) }, which took it from its own
// place k, and so on.  So with parent(v) = min { k > v : h(k) = v } every p[i]
// follows parents to their end, about e ln n of them at most.  The swaps that
// wrote to a place are listed by a counting sort.
#include "launch.h"

namespace tess {

namespace {

constexpr uint32_t kNone = 0xffffffffu;

// The (j + 1)-th output after state `seed` of splitmix64 (Steele, Lea and Flood).
__device__ uint64_t splitmix64_at(uint64_t seed, uint64_t j) {
  uint64_t z = seed + (j + 1) * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

__global__ __launch_bounds__(256) void k_shuffle_draw(uint64_t seed, uint32_t n, ShuffleBufs b) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const uint32_t h = i ? (uint32_t)(splitmix64_at(seed, n - 1 - i) % (i + 1)) : 0u;
  b.h[i] = h;
  b.rank[i] = i ? atomicAdd(&b.cnt[h], 1u) : kNone;  // place 0 has no swap of its own
}

__global__ __launch_bounds__(256) void k_shuffle_list(uint32_t n, ShuffleBufs b) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i < n && i) b.list[b.first[b.h[i]] + b.rank[i]] = i;
}

// The first swap after swap i (before it in k's order) that wrote to place v.
__device__ __forceinline__ uint32_t later(const ShuffleBufs& b, uint32_t v, uint32_t i) {
  uint32_t k = kNone;
  for (uint32_t q = b.first[v]; q < b.first[v + 1]; ++q) {
    const uint32_t s = b.list[q];
    k = s > i && s < k ? s : k;
  }
  return k;
}

// (parents take the ranks' place)
__global__ __launch_bounds__(256) void k_shuffle_parent(uint32_t n, ShuffleBufs b) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) b.rank[i] = later(b, i, i);
}

// Bound by the chains of dependent loads, 13 parents on average at their
// longest per wavefront; with the listing 400k samples take 70 us, on a
// host thread 980 us and 100 us of upload.
__global__ __launch_bounds__(256) void k_shuffle_walk(uint32_t n, ShuffleBufs b, int* __restrict__ p) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const uint32_t h = b.h[i];
  uint32_t k = h == i ? i : later(b, h, i);
  if (k == kNone) {
    p[i] = (int)h;
    return;
  }
  for (uint32_t q = b.rank[k]; q != kNone; q = b.rank[k]) k = q;
  p[i] = (int)k;
}

}  // namespace

hipError_t launch_shuffle(uint64_t* state, uint32_t n, const ShuffleBufs& b, int* p, hipStream_t s) {
  if (n == 0) return hipSuccess;
  const dim3 g((n + 255) / 256);
  hipError_t e = launch_fill_u32(b.cnt, n, 0u, s);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_shuffle_draw, g, dim3(256), 0, s, *state, n, b);
  if ((e = launch_scan_u32(b.cnt, (int)n, b.first, b.sums, b.first + n, s)) != hipSuccess) return e;
  hipLaunchKernelGGL(k_shuffle_list, g, dim3(256), 0, s, n, b);
  hipLaunchKernelGGL(k_shuffle_parent, g, dim3(256), 0, s, n, b);
  hipLaunchKernelGGL(k_shuffle_walk, g, dim3(256), 0, s, n, b, p);
  *state += (uint64_t)(n - 1) * 0x9E3779B97F4A7C15ull;
  return hipGetLastError();
}

}  // namespace tess
