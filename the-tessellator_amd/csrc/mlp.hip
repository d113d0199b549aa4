// mlp.hip -- the learned search-radius model: 27 -> 64 -> 64 -> 2 (ReLU),
// BF16 weights and activations on the MFMA units, FP32 accumulation.
//
// Features of a cell: log(1 + count) of the 27 grid cells around the site's
// grid cell (0 outside the grid), padded to 32.  Outputs (standardised):
// log(final R / smallest grid-cell edge) and log(1 + candidates streamed),
// as recorded by the plain kernel.
//
// Matrix products use v_mfma_f32_16x16x32_bf16: per wavefront
//   A (16 x 32): lane l holds row l&15, k = 8(l>>4) .. 8(l>>4)+7
//   B (32 x 16): lane l holds col l&15, k = 8(l>>4) .. 8(l>>4)+7
//   D (16 x 16): lane l holds col l&15, rows 4(l>>4) .. 4(l>>4)+3
// (checked by k_mfma_probe against a host product).
//
// The BF16 weights are kept twice: row-major, and as the fragments the
// products load (frag_pos), so that a B operand is one 16-byte load a lane
// instead of eight 2-byte ones a row apart.
//
// Training: one workgroup per 32 samples runs forward and backward; its
// weight gradients go to a slot of its own and k_adam reduces the slots in
// a fixed order (deterministic) and applies Adam to the FP32 master weights,
// refreshing the BF16 copies.
#include "launch.h"
#include "tess_internal.h"

namespace tess {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma(const bf16x8& a, const bf16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// round-to-nearest-even f32 -> bf16 bits
__device__ __forceinline__ uint16_t to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);  // NaN
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
// ReLU of four values as bf16 bits, rounded by the hardware conversion (ties
// to even like to_bf16; a NaN has become 0).
__device__ __forceinline__ uint2 relu4(const f32x4& z) {
  typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
  bf16x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = (__bf16)(z[i] > 0.f ? z[i] : 0.f);
  uint2 u;
  __builtin_memcpy(&u, &v, 8);
  return u;
}
__device__ __forceinline__ float from_bf16(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ __forceinline__ bf16x8 load8(const uint16_t* p) {
  bf16x8 v;
  __builtin_memcpy(&v, p, 16);
  return v;
}
// Four bf16 values as one 8-byte store.
__device__ __forceinline__ void store4(uint16_t* p, uint16_t a, uint16_t b, uint16_t c, uint16_t d) {
  *reinterpret_cast<uint2*>(p) = make_uint2((uint32_t)a | ((uint32_t)b << 16), (uint32_t)c | ((uint32_t)d << 16));
}
__device__ __forceinline__ bf16x8 gather8(const uint16_t* p, int stride) {
  uint16_t t[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) t[j] = p[j * stride];
  bf16x8 v;
  __builtin_memcpy(&v, t, 16);
  return v;
}

// Weight parameter i's place among the fragments: fragment f (W1: column
// block t; W2: 4 + 4 kk + t; W3: 12 + kk, kk the block of 32 inputs), then
// the lane that holds the column, then the input within the lane's eight.
__device__ __forceinline__ int frag_pos(int i) {
  int f, k, row;
  if (i < kMlpIn * kMlpH) {
    k = i / kMlpH;
    row = i % 16;
    f = (i % kMlpH) / 16;
  } else if (i < kMlpIn * kMlpH + kMlpH * kMlpH) {
    i -= kMlpIn * kMlpH;
    k = i / kMlpH;
    row = i % 16;
    f = 4 + 4 * (k / 32) + (i % kMlpH) / 16;
  } else {
    i -= kMlpIn * kMlpH + kMlpH * kMlpH;
    k = i / kMlpOutPad;
    row = i % kMlpOutPad;
    f = 12 + k / 32;
  }
  k %= 32;
  return (f * 64 + (k / 8) * 16 + row) * 8 + k % 8;
}

}  // namespace

// Lane-layout probe: D = A (16x32) * B (32x16), A and B given row-major.
__global__ __launch_bounds__(64) void k_mfma_probe(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                                                   float* __restrict__ D) {
  const int l = threadIdx.x, row = l & 15, kb = 8 * (l >> 4);
  const bf16x8 a = load8(A + row * 32 + kb);
  const bf16x8 b = gather8(B + kb * 16 + row, 16);
  f32x4 c = {0.f, 0.f, 0.f, 0.f};
  c = mfma(a, b, c);
#pragma unroll
  for (int i = 0; i < 4; ++i) D[(4 * (l >> 4) + i) * 16 + (l & 15)] = c[i];
}

// Features: log(1 + count) of the 3x3x3 grid cells around each point's grid
// cell (offsets -1..1, x outermost), 0 outside the grid; bf16, 32 per point
// (the last 5 are 0).  bins: grid cell of each point (original order); the
// points are taken in grid order, where neighbouring lanes read the same
// delimiters.  The
// values of counts below kFeatTab are computed once per workgroup into LDS by
// the same expression (so bit for bit the same) and looked up; a workgroup
// takes many points, so that the table's logarithms are few next to them.  A
// column of three grid cells is four delimiters in a row.  400k points: 54 ->
// 28 us (a table per 256 points, two delimiters per grid cell).
constexpr int kFeatTab = 1024;
__global__ __launch_bounds__(256) void k_features(const uint32_t* __restrict__ sorted,
                                                  const uint32_t* __restrict__ bins,
                                                  const uint32_t* __restrict__ delim, int cpd, int n,
                                                  uint16_t* __restrict__ feat) {
  __shared__ uint16_t tab[kFeatTab];
  for (int c = threadIdx.x; c < kFeatTab; c += blockDim.x) tab[c] = to_bf16((float)log1p((double)c));
  __syncthreads();
  auto value = [&](uint32_t c) { return c < (uint32_t)kFeatTab ? tab[c] : to_bf16((float)log1p((double)c)); };
  for (uint32_t k = blockIdx.x * 256u + threadIdx.x; k < (uint32_t)n; k += gridDim.x * 256u) {
    const uint32_t i = sorted[k];
    const int b0 = (int)bins[i];
    const int iz = b0 % cpd, iy = (b0 / cpd) % cpd, ix = b0 / (cpd * cpd);
    uint16_t f[kMlpIn] = {};
#pragma unroll
    for (int j = 0; j < 9; ++j) {
      const int bx = ix + j / 3 - 1, by = iy + j % 3 - 1;
      uint32_t d[4] = {0, 0, 0, 0};
      if (bx >= 0 && bx < cpd && by >= 0 && by < cpd) {
        const uint32_t* p = delim + ((bx * cpd + by) * cpd + iz);
        d[1] = p[0];
        d[2] = p[1];
        d[0] = iz > 0 ? p[-1] : d[1];
        d[3] = iz + 1 < cpd ? p[2] : d[2];
      }
#pragma unroll
      for (int z = 0; z < 3; ++z) f[3 * j + z] = value(d[z + 1] - d[z]);
    }
    uint4* dst = reinterpret_cast<uint4*>(feat + (size_t)i * kMlpIn);
    const uint4* src = reinterpret_cast<const uint4*>(f);
#pragma unroll
    for (int q = 0; q < kMlpIn / 8; ++q) dst[q] = src[q];
  }
}

// Forward (inference): a wavefront keeps every weight fragment in registers
// and takes 16 samples at a time; its activations pass through LDS of its
// own, rows padded to 72 values so that the 16-byte fragment reads spread
// over the banks.  out: 2 floats per sample (standardised).  400k samples:
// 38.7 -> 16.5 us (one wavefront per 16 samples re-read the 14 KB of weights
// two bytes at a time); what is left is latency of the chain of products.
constexpr int kRowH = kMlpH + 8;  // padded activation row
__global__ __launch_bounds__(256) void k_mlp_forward(const uint16_t* __restrict__ X, int n,
                                                     const uint16_t* __restrict__ WF, const float* __restrict__ bias,
                                                     float* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) uint16_t hs[4][16 * kRowH];
  const int l = threadIdx.x & 63, row = l & 15, kb = 8 * (l >> 4), r0 = 4 * (l >> 4);
  uint16_t* h = hs[threadIdx.x >> 6];
  auto sync = [] {  // the wavefront's LDS accesses stay in order
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  bf16x8 w[14];
#pragma unroll
  for (int f = 0; f < 14; ++f) w[f] = load8(WF + (f * 64 + l) * 8);
  float b1[4], b2[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    b1[t] = bias[16 * t + row];
    b2[t] = bias[kMlpH + 16 * t + row];
  }
  const float b3 = bias[2 * kMlpH + row];
  const uint32_t step = gridDim.x * 64u, count = (uint32_t)n;
  for (uint32_t s0 = (blockIdx.x * 4u + (threadIdx.x >> 6)) * 16u; s0 < count; s0 += step) {
    // layer 1: [16 x 32] x [32 x 64]
    bf16x8 a = {};
    if (s0 + row < count) a = load8(X + (size_t)(s0 + row) * kMlpIn + kb);
    f32x4 acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
      acc[t] = mfma(a, w[t], acc[t]);
    }
    sync();
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const uint2 v = relu4(acc[t] + b1[t]);
      uint16_t* p = h + r0 * kRowH + 16 * t + row;
      p[0] = (uint16_t)v.x;
      p[kRowH] = (uint16_t)(v.x >> 16);
      p[2 * kRowH] = (uint16_t)v.y;
      p[3 * kRowH] = (uint16_t)(v.y >> 16);
    }
    sync();
    // layer 2: [16 x 64] x [64 x 64]
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const bf16x8 ah = load8(h + row * kRowH + 32 * kk + kb);
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[t] = mfma(ah, w[4 + 4 * kk + t], acc[t]);
    }
    sync();
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const uint2 v = relu4(acc[t] + b2[t]);
      uint16_t* p = h + r0 * kRowH + 16 * t + row;
      p[0] = (uint16_t)v.x;
      p[kRowH] = (uint16_t)(v.x >> 16);
      p[2 * kRowH] = (uint16_t)v.y;
      p[3 * kRowH] = (uint16_t)(v.y >> 16);
    }
    sync();
    // layer 3: [16 x 64] x [64 x 16] (2 of 16 columns used)
    f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) y = mfma(load8(h + row * kRowH + 32 * kk + kb), w[12 + kk], y);
    if (row < kMlpOut)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (s0 + r0 + i < count) out[(size_t)(s0 + r0 + i) * kMlpOut + row] = y[i] + b3;
  }
}

// Forward + backward of 32 samples per workgroup of four wavefronts;
// mean-squared error over the whole batch (scale = 1 / batch).  Gradients of
// these samples go to grad + blockIdx.x * kMlpParams (the pad columns of W3
// and b3 are not written: the caller clears the slots once).
//
// Latency bounds it (a batch of 8,192 is one workgroup per CU): so the
// weight fragments are loaded while the samples' rows arrive, wavefront w
// takes samples 16 (w & 1) .. + 15 and column blocks 2 (w >> 1), + 1 in every
// product of the chain, pre-activations stay in the lanes that the backward
// pass needs them in, and activations are stored in both orders, so that
// every operand is one 16-byte LDS read.  8,192 samples: 35.5 -> 12.2 us
// (one wavefront per 32 samples, operands gathered two bytes at a time).
constexpr int kRowX = kMlpIn + 8, kRowS = 32 + 8;  // padded rows: features, samples
__global__ __launch_bounds__(256) void k_mlp_train_step(const uint16_t* __restrict__ X, const float* __restrict__ T,
                                                        const int* __restrict__ idx, int nsamp, float scale,
                                                        const uint16_t* __restrict__ W,
                                                        const float* __restrict__ bias, float* __restrict__ grad,
                                                        float* __restrict__ loss) {
  __shared__ __attribute__((aligned(16))) uint16_t xs[32 * kRowX], xT[kMlpIn * kRowS];
  __shared__ __attribute__((aligned(16))) uint16_t h1[32 * kRowH], h1T[kMlpH * kRowS];
  __shared__ __attribute__((aligned(16))) uint16_t h2[32 * kRowH], h2T[kMlpH * kRowS];
  __shared__ __attribute__((aligned(16))) uint16_t dz2[32 * kRowH], dz2T[kMlpH * kRowS], dz1T[kMlpH * kRowS];
  __shared__ float dy[32 * kMlpOut];
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, row = l & 15, kb = 8 * (l >> 4), r0 = 4 * (l >> 4);
  const int rb = 16 * (w & 1), t0 = 2 * (w >> 1);  // this wavefront's samples, its first column block
  const int s0 = blockIdx.x * 32;
  const uint16_t *W2 = W + kMlpIn * kMlpH, *W3 = W2 + kMlpH * kMlpH, *WF = W + kMlpWeights;
  float* g = grad + (size_t)blockIdx.x * kMlpParams;
  float *gW1 = g, *gW2 = g + kMlpIn * kMlpH, *gW3 = gW2 + kMlpH * kMlpH, *gb1 = gW3 + kMlpH * kMlpOutPad,
        *gb2 = gb1 + kMlpH, *gb3 = gb2 + kMlpH;
  // the samples' features (zero rows past the end), four a thread
  const int ss = tid >> 3, part = 4 * (tid & 7);
  uint2 xv = make_uint2(0, 0);
  if (s0 + ss < nsamp) xv = *reinterpret_cast<const uint2*>(X + (size_t)idx[s0 + ss] * kMlpIn + part);
  // weights of this wavefront's tiles, forward and (W2) backward
  bf16x8 w1[2], w2[2][2], w2b[2][2], w3[2];
  float b1[2], b2[2], w3o[2][kMlpOut];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int col = 16 * (t0 + t) + row;
    w1[t] = load8(WF + ((t0 + t) * 64 + l) * 8);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      w2[kk][t] = load8(WF + ((4 + 4 * kk + t0 + t) * 64 + l) * 8);
      w2b[t][kk] = load8(W2 + col * kMlpH + 32 * kk + kb);
    }
    b1[t] = bias[col];
    b2[t] = bias[kMlpH + col];
#pragma unroll
    for (int o = 0; o < kMlpOut; ++o) w3o[t][o] = from_bf16(W3[col * kMlpOutPad + o]);
  }
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) w3[kk] = load8(WF + ((12 + kk) * 64 + l) * 8);
  const float b3 = bias[2 * kMlpH + row];
  float tv[2][4];  // wavefront 0: this lane's targets
  if (w == 0 && row < kMlpOut)
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int s = 16 * half + r0 + i;
        tv[half][i] = s0 + s < nsamp ? T[(size_t)idx[s0 + s] * kMlpOut + row] : 0.f;
      }
  *reinterpret_cast<uint2*>(xs + ss * kRowX + part) = xv;
  xT[part * kRowS + ss] = (uint16_t)xv.x;
  xT[(part + 1) * kRowS + ss] = (uint16_t)(xv.x >> 16);
  xT[(part + 2) * kRowS + ss] = (uint16_t)xv.y;
  xT[(part + 3) * kRowS + ss] = (uint16_t)(xv.y >> 16);
  __syncthreads();
  // forward: pre-activations stay in registers, ReLU outputs go to LDS by
  // sample and by unit
  f32x4 z1[2], z2[2];
  auto activate = [&](f32x4 (&z)[2], const float (&b)[2], uint16_t* h, uint16_t* hT) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int col = 16 * (t0 + t) + row;
      z[t] = z[t] + b[t];
      const uint2 v = relu4(z[t]);
      uint16_t* p = h + (rb + r0) * kRowH + col;
      p[0] = (uint16_t)v.x;
      p[kRowH] = (uint16_t)(v.x >> 16);
      p[2 * kRowH] = (uint16_t)v.y;
      p[3 * kRowH] = (uint16_t)(v.y >> 16);
      *reinterpret_cast<uint2*>(hT + col * kRowS + rb + r0) = v;
    }
  };
  {
    const bf16x8 a = load8(xs + (rb + row) * kRowX + kb);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      z1[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
      z1[t] = mfma(a, w1[t], z1[t]);
    }
  }
  activate(z1, b1, h1, h1T);
  __syncthreads();
#pragma unroll
  for (int t = 0; t < 2; ++t) z2[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    const bf16x8 ah = load8(h1 + (rb + row) * kRowH + 32 * kk + kb);
#pragma unroll
    for (int t = 0; t < 2; ++t) z2[t] = mfma(ah, w2[kk][t], z2[t]);
  }
  activate(z2, b2, h2, h2T);
  __syncthreads();
  // output layer, dL/dy and the loss: wavefront 0, both halves in turn (the
  // loss adds up in a fixed order)
  float lsum = 0.f;
  if (w == 0) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) y = mfma(load8(h2 + (16 * half + row) * kRowH + 32 * kk + kb), w3[kk], y);
      if (row < kMlpOut)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int s = 16 * half + r0 + i;
          float d = 0.f;
          if (s0 + s < nsamp) {
            const float diff = y[i] + b3 - tv[half][i];
            d = diff * scale;
            lsum += 0.5f * diff * diff;
          }
          dy[s * kMlpOut + row] = d;
        }
    }
  }
  __syncthreads();
  // dz2 = (dy W3^T) * [z2 > 0]
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int col = 16 * (t0 + t) + row;
    uint16_t v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float d = 0.f;
#pragma unroll
      for (int o = 0; o < kMlpOut; ++o) d += dy[(rb + r0 + i) * kMlpOut + o] * w3o[t][o];
      v[i] = to_bf16(z2[t][i] > 0.f ? d : 0.f);
      dz2[(rb + r0 + i) * kRowH + col] = v[i];
    }
    store4(dz2T + col * kRowS + rb + r0, v[0], v[1], v[2], v[3]);
  }
  // dW3 = h2^T dy, db3 = sum dy (VALU: 64 x 2 outputs over 32 samples)
  if (tid < kMlpH * kMlpOut) {
    const int hi = tid / kMlpOut, o = tid % kMlpOut;
    float s = 0.f;
#pragma unroll
    for (int q = 0; q < 32; ++q) s += from_bf16(h2T[hi * kRowS + q]) * dy[q * kMlpOut + o];
    gW3[hi * kMlpOutPad + o] = s;
  } else if (tid < kMlpH * kMlpOut + kMlpOut) {
    const int o = tid - kMlpH * kMlpOut;
    float s = 0.f;
    for (int q = 0; q < 32; ++q) s += dy[q * kMlpOut + o];
    gb3[o] = s;
  }
  __syncthreads();
  // dz1 = (dz2 W2^T) * [z1 > 0]  (K = 64)
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    f32x4 dh = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) dh = mfma(load8(dz2 + (rb + row) * kRowH + 32 * kk + kb), w2b[t][kk], dh);
    uint16_t v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = to_bf16(z1[t][i] > 0.f ? dh[i] : 0.f);
    store4(dz1T + (16 * (t0 + t) + row) * kRowS + rb + r0, v[0], v[1], v[2], v[3]);
  }
  // dW2 = h1^T dz2 (K = 32 samples), db2 = sum dz2: wavefront w takes units
  // 16 w .. + 15 of layer 1
  {
    const bf16x8 a = load8(h1T + (16 * w + row) * kRowS + kb);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      f32x4 c = {0.f, 0.f, 0.f, 0.f};
      c = mfma(a, load8(dz2T + (16 * t + row) * kRowS + kb), c);
#pragma unroll
      for (int i = 0; i < 4; ++i) gW2[(16 * w + r0 + i) * kMlpH + 16 * t + row] = c[i];
    }
  }
  if (w == 3) {
    float s = 0.f;
#pragma unroll
    for (int q = 0; q < 32; ++q) s += from_bf16(dz2T[l * kRowS + q]);
    gb2[l] = s;
  }
  __syncthreads();
  // dW1 = x^T dz1 (K = 32 samples), db1 = sum dz1
  {
    const int m = w & 1;
    const bf16x8 a = load8(xT + (16 * m + row) * kRowS + kb);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      f32x4 c = {0.f, 0.f, 0.f, 0.f};
      c = mfma(a, load8(dz1T + (16 * (t0 + t) + row) * kRowS + kb), c);
#pragma unroll
      for (int i = 0; i < 4; ++i) gW1[(16 * m + r0 + i) * kMlpH + 16 * (t0 + t) + row] = c[i];
    }
  }
  if (w == 3) {
    float s = 0.f;
#pragma unroll
    for (int q = 0; q < 32; ++q) s += from_bf16(dz1T[l * kRowS + q]);
    gb1[l] = s;
  }
  // the workgroup's loss
  if (w == 0) {
    for (int o = 32; o > 0; o >>= 1) lsum += __shfl_xor(lsum, o, 64);
    if (l == 0) loss[blockIdx.x] = lsum;
  }
}

// Sum of nslots gradient slots of parameter i in slot order, the same on
// every wavefront of the workgroup (64 parameters, one a lane).  A running
// sum has to stay in order, its loads do not: each of the four wavefronts
// has 64 slots in flight, then they add theirs in turn, the sum passing
// through LDS.
__device__ __forceinline__ float slot_sum(const float* __restrict__ grad, int nslots, int i, bool live) {
  __shared__ float run[64];
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (w == 0) run[l] = 0.f;
  for (int base = 0; base < nslots; base += 256) {
    const int b = base + 64 * w;
    const int m = nslots - b < 64 ? nslots - b : 64;  // this wavefront's slots (<= 0: none)
    float v[64];
    if (live && m == 64) {
#pragma unroll
      for (int k = 0; k < 64; ++k) v[k] = grad[(size_t)(b + k) * kMlpParams + i];
    } else if (live) {
#pragma unroll
      for (int k = 0; k < 64; ++k)
        if (k < m) v[k] = grad[(size_t)(b + k) * kMlpParams + i];
    }
    for (int turn = 0; turn < 4; ++turn) {
      __syncthreads();
      if (w == turn && live && m > 0) {
        float s = run[l];
        if (m == 64) {
#pragma unroll
          for (int k = 0; k < 64; ++k) s += v[k];
        } else {
#pragma unroll
          for (int k = 0; k < 64; ++k)
            if (k < m) s += v[k];
        }
        run[l] = s;
      }
    }
  }
  __syncthreads();
  return run[l];
}

// The bf16 copies (row-major, fragments) and the fp32 bias of parameter i.
__device__ __forceinline__ void store_param(int i, float w, uint16_t* __restrict__ wbf, float* __restrict__ bias) {
  if (i < kMlpWeights) {
    const uint16_t h = to_bf16(w);
    wbf[i] = h;
    wbf[kMlpWeights + frag_pos(i)] = h;
  } else {
    bias[i - kMlpWeights] = w;
  }
}

// Adam on the FP32 master parameters; gradients are the sum of nslots
// slots, added in slot order.  Refreshes the bf16 weights.  256 slots: 58.8 ->
// 4.8 us (one thread per parameter read its slots one after another).
__global__ __launch_bounds__(256) void k_adam(const float* __restrict__ grad, int nslots, float* __restrict__ master,
                                              float* __restrict__ m1, float* __restrict__ m2,
                                              uint16_t* __restrict__ wbf, float* __restrict__ bias, float lr,
                                              float b1c, float b2c) {
  const int i = blockIdx.x * 64 + (threadIdx.x & 63);
  const float gsum = slot_sum(grad, nslots, i, i < kMlpParams);
  if (i >= kMlpParams || threadIdx.x >= 64) return;
  const float beta1 = 0.9f, beta2 = 0.999f, eps = 1e-8f;
  m1[i] = beta1 * m1[i] + (1.f - beta1) * gsum;
  m2[i] = beta2 * m2[i] + (1.f - beta2) * gsum * gsum;
  const float mh = m1[i] / b1c, vh = m2[i] / b2c;
  const float w = master[i] - lr * mh / (sqrtf(vh) + eps);
  master[i] = w;
  store_param(i, w, wbf, bias);
}

// Training targets from the plain search's counters: log(R / s_min) with R
// the final security radius, and log(1 + classified candidates); vmax: the
// largest vertex count the cell reached (at least 65 when the cell had to be
// rerun at a larger capacity: its cuts ran out of the 64 slots).
__global__ void k_targets(const tess_cell_stats* __restrict__ st, int n, double smin, float* __restrict__ T,
                          uint16_t* __restrict__ vmax) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const tess_cell_stats c = st[i];
  T[2 * i] = (float)log(sqrt(c.r2) / smin);
  T[2 * i + 1] = (float)log1p((double)c.classified);
  uint32_t v = c.max_vertices < 65535u ? c.max_vertices : 65535u;
  if ((c.status & TESS_CELL_RERUN) && v < 65u) v = 65u;
  vmax[i] = (uint16_t)v;
}

// Sum of nslots gradient slots in slot order.
__global__ __launch_bounds__(256) void k_grad_sum(const float* __restrict__ grad, int nslots,
                                                  float* __restrict__ out) {
  const int i = blockIdx.x * 64 + (threadIdx.x & 63);
  const float g = slot_sum(grad, nslots, i, i < kMlpParams);
  if (i < kMlpParams && threadIdx.x < 64) out[i] = g;
}

// Per column the sum of T, or of (T - mean)^2 when the blocks' sums are given:
// 256 blocks, each thread a strided row sum, then a tree.  Bound by latency:
// 400k rows 16 us for both and the end, 720 us on a host thread with the
// download.
__device__ double block_sum(double v, double* lds) {
  lds[threadIdx.x] = v;
  __syncthreads();
  for (int m = 128; m > 0; m >>= 1) {
    if ((int)threadIdx.x < m) lds[threadIdx.x] += lds[threadIdx.x + m];
    __syncthreads();
  }
  const double r = lds[0];
  __syncthreads();
  return r;
}

__global__ __launch_bounds__(256) void k_moments(const float* __restrict__ T, size_t n,
                                                 const double* __restrict__ sums, double* __restrict__ out) {
  __shared__ double lds[256];
  double mean[2] = {0, 0};
  if (sums)
    for (int k = 0; k < 2; ++k) mean[k] = block_sum(sums[2 * threadIdx.x + k], lds) / (double)n;
  double a[2] = {0, 0};
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)kMomentBlocks * 256)
    for (int k = 0; k < 2; ++k) {
      const double v = T[2 * i + k];
      a[k] += sums ? (v - mean[k]) * (v - mean[k]) : v;
    }
  for (int k = 0; k < 2; ++k) {
    const double r = block_sum(a[k], lds);
    if (threadIdx.x == 0) out[2 * blockIdx.x + k] = r;
  }
}

__global__ __launch_bounds__(256) void k_moments_end(double* __restrict__ part) {
  __shared__ double lds[256];
  double r[4];
  for (int k = 0; k < 4; ++k) r[k] = block_sum(part[2 * kMomentBlocks * (k >> 1) + 2 * threadIdx.x + (k & 1)], lds);
  if (threadIdx.x == 0)
    for (int k = 0; k < 4; ++k) part[k] = r[k];
}

// Standardise targets: Tn = (T - mean) / std per column.
__global__ void k_standardise(const float* __restrict__ T, size_t n, float m0, float s0, float m1, float s1,
                              float* __restrict__ Tn) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  Tn[2 * i] = (T[2 * i] - m0) / s0;
  Tn[2 * i + 1] = (T[2 * i + 1] - m1) / s1;
}

// bf16 copies of the weight part of the master parameters; biases to fp32.
__global__ void k_weights_from_master(const float* __restrict__ master, uint16_t* __restrict__ wbf,
                                      float* __restrict__ bias) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < kMlpParams) store_param(i, master[i], wbf, bias);
}

// Predicted radius (length units) and classified candidates of every point
// from the network's standardised outputs, in double like the targets.
// 400k points: 4 us (one exponential after the other on the host took
// about 5 ms).
__global__ __launch_bounds__(256) void k_predictions(const float* __restrict__ y, int n, PredictScale p,
                                                     float* __restrict__ out) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= (uint32_t)n) return;
  const float2 v = reinterpret_cast<const float2*>(y)[i];
  reinterpret_cast<float2*>(out)[i] = make_float2((float)(exp((double)v.x * p.norm[1] + p.norm[0]) * p.smin),
                                                  (float)expm1((double)v.y * p.norm[3] + p.norm[2]));
}

// Samples by their predicted log(1 + C) (bins of 1/4, kCalibBins of them):
// hist[0][b] all, hist[1 + r][b] those that outgrew 64 << r vertices.
__global__ __launch_bounds__(256) void k_calibration(const float* __restrict__ y, const uint16_t* __restrict__ vmax,
                                                     size_t n, float scale, float shift, uint32_t* __restrict__ hist) {
  __shared__ uint32_t h[3 * kCalibBins];
  for (int k = threadIdx.x; k < 3 * kCalibBins; k += 256) h[k] = 0;
  __syncthreads();
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    const float f = floorf((y[2 * i + 1] * scale + shift) * 4.0f);
    // a value no int holds (NaN among them) counts with the smallest
    const int b = fabsf(f) < 2147483648.0f ? (int)f : 0;
    const int bin = b < 0 ? 0 : (b < kCalibBins ? b : kCalibBins - 1);
    atomicAdd(&h[bin], 1u);
    if (vmax[i] > 64) atomicAdd(&h[kCalibBins + bin], 1u);
    if (vmax[i] > 128) atomicAdd(&h[2 * kCalibBins + bin], 1u);
  }
  __syncthreads();
  for (int k = threadIdx.x; k < 3 * kCalibBins; k += 256)
    if (h[k]) atomicAdd(&hist[k], h[k]);
}

hipError_t launch_predictions(const float* y, int n, const PredictScale& p, float* out, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_predictions, dim3((n - 1) / 256 + 1), dim3(256), 0, s, y, n, p, out);
  return hipGetLastError();
}

hipError_t launch_calibration(const float* y, const uint16_t* vmax, size_t n, float scale, float shift,
                              uint32_t* hist, hipStream_t s) {
  if (n == 0) return hipSuccess;
  const size_t blocks = (n + 255) / 256;
  hipLaunchKernelGGL(k_calibration, dim3((unsigned)(blocks < 512 ? blocks : 512)), dim3(256), 0, s, y, vmax, n, scale,
                     shift, hist);
  return hipGetLastError();
}

hipError_t launch_targets(const tess_cell_stats* st, int n, double smin, float* T, uint16_t* vmax, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_targets, dim3((n + 255) / 256), dim3(256), 0, s, st, n, smin, T, vmax);
  return hipGetLastError();
}

hipError_t launch_grad_sum(const float* grad, int nslots, float* out, hipStream_t s) {
  hipLaunchKernelGGL(k_grad_sum, dim3((kMlpParams + 63) / 64), dim3(256), 0, s, grad, nslots, out);
  return hipGetLastError();
}

hipError_t launch_moments(const float* T, size_t n, double* part, double out[4], hipStream_t s) {
  static_assert(kMomentBlocks == 256, "a block's sum per thread");
  double* part2 = part + 2 * kMomentBlocks;
  hipLaunchKernelGGL(k_moments, dim3(kMomentBlocks), dim3(256), 0, s, T, n, (const double*)nullptr, part);
  hipLaunchKernelGGL(k_moments, dim3(kMomentBlocks), dim3(256), 0, s, T, n, (const double*)part, part2);
  hipLaunchKernelGGL(k_moments_end, dim3(1), dim3(256), 0, s, part);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(out, part, 32, hipMemcpyDeviceToHost, s);
  return e == hipSuccess ? hipStreamSynchronize(s) : e;
}

hipError_t launch_standardise(const float* T, size_t n, const float norm[4], float* Tn, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_standardise, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, T, n, norm[0], norm[1],
                     norm[2], norm[3], Tn);
  return hipGetLastError();
}

hipError_t launch_weights_from_master(const float* master, uint16_t* wbf, float* bias, hipStream_t s) {
  hipLaunchKernelGGL(k_weights_from_master, dim3((kMlpParams + 255) / 256), dim3(256), 0, s, master, wbf, bias);
  return hipGetLastError();
}

hipError_t launch_mfma_probe(const uint16_t* A, const uint16_t* B, float* D, hipStream_t s) {
  hipLaunchKernelGGL(k_mfma_probe, dim3(1), dim3(64), 0, s, A, B, D);
  return hipGetLastError();
}

hipError_t launch_features(const uint32_t* sorted, const uint32_t* bins, const uint32_t* delim, int cpd, int n, uint16_t* feat,
                           hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int blocks = (n - 1) / 256 + 1;
  hipLaunchKernelGGL(k_features, dim3(blocks < 1024 ? blocks : 1024), dim3(256), 0, s, sorted, bins, delim, cpd, n, feat);
  return hipGetLastError();
}

hipError_t launch_mlp_forward(const uint16_t* X, int n, const uint16_t* W, const float* bias, float* out,
                              hipStream_t s) {
  if (n <= 0) return hipSuccess;
  // enough workgroups for every CU's wavefront slots; each loops over its samples
  const int blocks = (n - 1) / 64 + 1;
  hipLaunchKernelGGL(k_mlp_forward, dim3(blocks < 1024 ? blocks : 1024), dim3(256), 0, s, X, n, W + kMlpWeights, bias,
                     out);
  return hipGetLastError();
}

hipError_t launch_mlp_train_step(const uint16_t* X, const float* T, const int* idx, int nsamp, float scale,
                                 const uint16_t* W, const float* bias, float* grad, float* loss, hipStream_t s) {
  hipLaunchKernelGGL(k_mlp_train_step, dim3((nsamp + 31) / 32), dim3(256), 0, s, X, T, idx, nsamp, scale, W, bias,
                     grad, loss);
  return hipGetLastError();
}

hipError_t launch_adam(const float* grad, int nslots, float* master, float* m1, float* m2, uint16_t* wbf,
                       float* bias, float lr, float b1c, float b2c, hipStream_t s) {
  hipLaunchKernelGGL(k_adam, dim3((kMlpParams + 63) / 64), dim3(256), 0, s, grad, nslots, master, m1, m2, wbf, bias,
                     lr, b1c, b2c);
  return hipGetLastError();
}

}  // namespace tess
