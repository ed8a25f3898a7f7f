// Row-wise passes of a hybrid model's step of few rows, straight from the split sums of the product before them
// (fp32, as linear_rows leaves them). First the residual epilogue, a [SA, T, W], b [SB, T, W]:
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

// What a parallel sublayer's input product, as split sums part [S, T, N], is wanted for, in one pass: sums (+ bias), then
// left q rotated in pairs and rounded, left k rotated into the cache with itself as the value, head gates and the right
// gate rounded, and silu of the right q, k, v in the recurrence's order. Four columns a thread; at: first columns of left
// q, k, head gates and right q, k, v, gate, all multiples of 8.
//
// Bound by the sums' bytes (5.6 MB for 40 rows of 8720 in 4 shares) and a launch. In place of a product in one share (21 us
// of it), the rotation's pass and the silu pass (8 us): a step of 40 rows 699 us before, 678 with it, of 2 rows 635 and 586.
struct SplitColumns { int at[7]; };

__global__ void __launch_bounds__(256) hybrid_split_kernel(
    const float* __restrict__ part, int S, const bfraw* __restrict__ bias, SplitColumns cols,
    const int64_t* __restrict__ positions, const float* __restrict__ inv_freq, bfraw* __restrict__ k_cache,
    bfraw* __restrict__ v_cache, const int64_t* __restrict__ slots, bfraw* __restrict__ q_out,
    bfraw* __restrict__ head_gate, float* __restrict__ packed, bfraw* __restrict__ gate, int T_, int N, int H, int G,
    int R, int BS, int RH, int RD, int RV) {
  const int t = blockIdx.y, c = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (c >= N) return;
  float x[4] = {};
  const float* p = part + (int64_t)t * N + c;
#pragma unroll 4
  for (int s = 0; s < S; ++s) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(p + (int64_t)s * T_ * N);
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] += v[e];
  }
  if (bias) {
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] += ldf(bias + c + e);
  }
  auto put = [](bfraw* o, const float (&v)[4]) {
    *reinterpret_cast<uint2*>(o) = make_uint2(bf_bits(v[0]) | (bf_bits(v[1]) << 16), bf_bits(v[2]) | (bf_bits(v[3]) << 16));
  };
  auto in = [&](int i, int n) { return c >= cols.at[i] && c < cols.at[i] + n; };
  const bool is_q = in(0, H * 128);
  if (is_q || in(1, G * 128)) {
    const int o = c - cols.at[is_q ? 0 : 1], dim = o % 128;
    float y[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float sn = 0.0f, cs = 1.0f;
      if (dim / 2 + i < R) sincosf((float)positions[t] * inv_freq[dim / 2 + i], &sn, &cs);
      y[2 * i] = x[2 * i] * cs - x[2 * i + 1] * sn;
      y[2 * i + 1] = x[2 * i + 1] * cs + x[2 * i] * sn;
    }
    if (is_q) {
      put(q_out + (int64_t)t * H * 128 + o, y);
    } else {
      const int64_t slot = slots[t], row = (slot / BS * G + o / 128) * BS + slot % BS;
      put(k_cache + row * 128 + dim, y);
      put(v_cache + row * 128 + dim, x);
    }
  } else if (in(2, H)) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (c + e < cols.at[2] + H) stf(head_gate + (int64_t)t * H + c - cols.at[2] + e, x[e]);
  } else if (in(6, RH * RV)) {
    put(gate + (int64_t)t * RH * RV + c - cols.at[6], x);
  } else {
#pragma unroll
    for (int i = 3; i < 6; ++i) {
      const int w = i == 5 ? RV : RD;    // a multiple of 4
      if (!in(i, RH * w)) continue;
      const int o = c - cols.at[i], h = o / w;
      float* to = packed + ((int64_t)t * RH + h) * (2 * RD + RV) + (i - 3) * RD + o % w;
      f32x4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = silu_exact(x[e]);
      *reinterpret_cast<f32x4*>(to) = y;
    }
  }
}

extern "C" void seq_launch_hybrid_split(const float* part, int S, const void* bias, const int64_t* at,
                                        const int64_t* positions, const float* inv_freq, void* k_cache, void* v_cache,
                                        const int64_t* slots, void* q_out, void* head_gate, float* packed, void* gate,
                                        int T_, int N, int H, int G, int R, int BS, int RH, int RD, int RV,
                                        hipStream_t st) {
  SplitColumns cols;
  for (int i = 0; i < 7; ++i) cols.at[i] = (int)at[i];
  hipLaunchKernelGGL(hybrid_split_kernel, dim3((N / 4 + 255) / 256, T_), dim3(256), 0, st, part, S, (const bfraw*)bias,
                     cols, positions, inv_freq, (bfraw*)k_cache, (bfraw*)v_cache, slots, (bfraw*)q_out, (bfraw*)head_gate,
                     packed, (bfraw*)gate, T_, N, H, G, R, BS, RH, RD, RV);
}
