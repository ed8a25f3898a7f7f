// The residual epilogue of a step of few rows, straight from the split sums of the product before it (a [SA, T, W],
// b [SB, T, W] fp32, as linear_rows leaves them):
//   y = a, or (rms(a) wa + rms(b) wb) / 2;  x += rms(y) w_post;  out = rms(x) w_next in bf16
//
// A row is one workgroup's: its sums are the bytes, 64 to 128 KB of them, and the three reductions the chain behind. Four
// columns a thread and load, kept in registers through all passes. 40 rows of 2048 in 8 shares: 5.2 us
// of a step, 7.8 with two branches (4.8 and 6.5 from bf16 products, which took 12 and 12 to 17 us themselves, 5.3 now).

#include "seq_common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define SR_THREADS 512
#define SR_VECS 4          // W <= 4 * 4 * 512

template <bool DUAL>
__global__ void __launch_bounds__(SR_THREADS) sandwich_rows_kernel(
    float* __restrict__ x, const float* __restrict__ a, int SA, const float* __restrict__ b, int SB,
    const float* __restrict__ wa, const float* __restrict__ wb, const float* __restrict__ w_post,
    const float* __restrict__ w_next, bfraw* __restrict__ out, int T_, int W, float eps) {
  __shared__ float scratch[16];
  const int t = blockIdx.x, tid = threadIdx.x, nvec = W / 4;
  const int64_t plane = (int64_t)T_ * W;
  const float inv_w = 1.0f / (float)W;
  auto sums = [&](const float* p, int S, f32x4 (&v)[SR_VECS]) {
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < SR_VECS; ++k) {
      v[k] = f32x4{0.f, 0.f, 0.f, 0.f};
      const int i = tid + k * SR_THREADS;
      if (i >= nvec) break;
      const float* q = p + (int64_t)t * W + i * 4;
#pragma unroll 8
      for (int s = 0; s < S; ++s) {
        const f32x4 u = *reinterpret_cast<const f32x4*>(q + s * plane);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[k][e] += u[e];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) ss += v[k][e] * v[k][e];
    }
    return ss;
  };
  f32x4 y[SR_VECS];
  float ss = sums(a, SA, y);
  if constexpr (DUAL) {
    f32x4 z[SR_VECS];
    const float sb = sums(b, SB, z);
    const float ra = 1.0f / sqrtf(block_sum(ss, scratch) * inv_w + eps);
    const float rb = 1.0f / sqrtf(block_sum(sb, scratch) * inv_w + eps);
    ss = 0.0f;
#pragma unroll
    for (int k = 0; k < SR_VECS; ++k) {
      const int i = tid + k * SR_THREADS;
      if (i >= nvec) break;
      const f32x4 ga = reinterpret_cast<const f32x4*>(wa)[i], gb = reinterpret_cast<const f32x4*>(wb)[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        y[k][e] = 0.5f * (y[k][e] * ra * ga[e] + z[k][e] * rb * gb[e]);
        ss += y[k][e] * y[k][e];
      }
    }
  }
  const float ry = 1.0f / sqrtf(block_sum(ss, scratch) * inv_w + eps);
  float sx = 0.0f;
#pragma unroll
  for (int k = 0; k < SR_VECS; ++k) {
    const int i = tid + k * SR_THREADS;
    if (i >= nvec) break;
    f32x4* px = reinterpret_cast<f32x4*>(x + (int64_t)t * W) + i;
    const f32x4 old = *px, g = reinterpret_cast<const f32x4*>(w_post)[i];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      y[k][e] = old[e] + y[k][e] * ry * g[e];
      sx += y[k][e] * y[k][e];
    }
    *px = y[k];
  }
  const float rx = 1.0f / sqrtf(block_sum(sx, scratch) * inv_w + eps);
#pragma unroll
  for (int k = 0; k < SR_VECS; ++k) {
    const int i = tid + k * SR_THREADS;
    if (i >= nvec) break;
    const f32x4 g = reinterpret_cast<const f32x4*>(w_next)[i];
    uint2 o;
    o.x = bf_bits(y[k][0] * rx * g[0]) | (bf_bits(y[k][1] * rx * g[1]) << 16);
    o.y = bf_bits(y[k][2] * rx * g[2]) | (bf_bits(y[k][3] * rx * g[3]) << 16);
    reinterpret_cast<uint2*>(out + (int64_t)t * W)[i] = o;
  }
}

// b nullptr: one branch
extern "C" void seq_launch_sandwich_rows(float* x, const float* a, int SA, const float* b, int SB, const float* wa,
                                         const float* wb, const float* w_post, const float* w_next, void* out, int T_,
                                         int W, float eps, hipStream_t st) {
  if (b)
    hipLaunchKernelGGL(sandwich_rows_kernel<true>, dim3(T_), dim3(SR_THREADS), 0, st, x, a, SA, b, SB, wa, wb, w_post,
                       w_next, (bfraw*)out, T_, W, eps);
  else
    hipLaunchKernelGGL(sandwich_rows_kernel<false>, dim3(T_), dim3(SR_THREADS), 0, st, x, a, SA, b, SB, wa, wb, w_post,
                       w_next, (bfraw*)out, T_, W, eps);
}
