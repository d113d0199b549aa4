// copyout.hip -- results to the host: the device writes several arrays into
// pinned host memory in one pass.
#include "launch.h"

namespace tess {

namespace {

constexpr int kCopyUnits = 4;  // 16-byte units of a lane in flight

// Bytes [base, base + len) of the pieces laid end to end (each from a
// multiple of 16) into dst.  Bound by the link to the host (55 GB/s for 16 MiB and
// more); below that by what a transfer costs before it starts, which is why
// all arrays of a call go in one launch (a hipMemcpy each to pageable memory:
// 15 us, and 17 GB/s for large ones).  A call with its downloads, before and
// after: a single cell 231 -> 137 us, 64 sets of a batch 28.0 -> 22.0 ms,
// cells and geometry of 100k points 7.2 -> 5.8 ms.  Stores are 1 KiB per wavefront and
// in order; sources are read in 16 bytes where their alignment allows, a
// piece's last bytes one by one (nothing is read past its end).
__global__ __launch_bounds__(256) void k_copy_out(CopyOut a) {
  const uint64_t units = (a.len + 15) / 16, stride = (uint64_t)gridDim.x * 256;
  for (uint64_t u0 = (uint64_t)blockIdx.x * 256 + threadIdx.x; u0 < units; u0 += stride * kCopyUnits) {
    uint4 w[kCopyUnits];
#pragma unroll
    for (int k = 0; k < kCopyUnits; ++k) {
      const uint64_t u = u0 + k * stride;
      if (u >= units) break;
      const uint64_t v = a.base + 16 * u;
      int p = 0;
      for (int q = 1; q < a.npieces; ++q)
        if (v >= a.piece[q].start) p = q;
      const CopyOutPiece& P = a.piece[p];
      const uint64_t off = v - P.start;
      const char* src = static_cast<const char*>(P.src) + off;
      const uintptr_t al = reinterpret_cast<uintptr_t>(src);
      w[k] = make_uint4(0, 0, 0, 0);
      if (off + 16 <= P.bytes && (al & 15) == 0) {
        w[k] = *reinterpret_cast<const uint4*>(src);
      } else if (off + 16 <= P.bytes && (al & 3) == 0) {
        const uint32_t* s = reinterpret_cast<const uint32_t*>(src);
        w[k] = make_uint4(s[0], s[1], s[2], s[3]);
      } else if (off < P.bytes) {
        uint32_t t[4] = {0, 0, 0, 0};
#pragma unroll
        for (int b = 0; b < 16; ++b)
          if (off + b < P.bytes) t[b >> 2] |= (uint32_t)(uint8_t)src[b] << (8 * (b & 3));
        w[k] = make_uint4(t[0], t[1], t[2], t[3]);
      }
      if (P.sub) {
        const uint64_t m = *P.sub;
        const uint64_t x = (((uint64_t)w[k].y << 32) | w[k].x) - m, y = (((uint64_t)w[k].w << 32) | w[k].z) - m;
        w[k] = make_uint4((uint32_t)x, (uint32_t)(x >> 32), (uint32_t)y, (uint32_t)(y >> 32));
      }
    }
#pragma unroll
    for (int k = 0; k < kCopyUnits; ++k) {
      const uint64_t u = u0 + k * stride;
      if (u >= units) break;
      reinterpret_cast<uint4*>(a.dst)[u] = w[k];
    }
  }
}

// out[k] = src[at[k]]
__global__ __launch_bounds__(256) void k_pick_u64(const uint64_t* __restrict__ src, const uint64_t* __restrict__ at,
                                                  int n, uint64_t* __restrict__ out) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k < n) out[k] = src[at[k]];
}

}  // namespace

hipError_t launch_copy_out(const CopyOut& a, hipStream_t s) {
  if (a.len == 0) return hipSuccess;
  const uint64_t blocks = (a.len + 16 * 256 * kCopyUnits - 1) / (16 * 256 * kCopyUnits);
  hipLaunchKernelGGL(k_copy_out, dim3((unsigned)(blocks < 1024 ? blocks : 1024)), dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_pick_u64(const uint64_t* src, const uint64_t* at, int n, uint64_t* out, hipStream_t s) {
  hipLaunchKernelGGL(k_pick_u64, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, src, at, n, out);
  return hipGetLastError();
}

}  // namespace tess
