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

// A gated-delta-rule sublayer between its input product (split sums part [S, T, N]) and its output product, single tokens:
// convolution and silu of q, k, v with the carried history, the two low-rank products, decay and write strength, the step of
// the recurrence, the gated norm of each head. A workgroup is a row's key head with the heads that share it, so a channel's
// history has one reader and writer. Rounded where the general sublayer's launches round: inputs, convolved values, low-rank
// products and the result to bf16.
//
// Bound by the state's bytes (512 KB a row, read and written) and the chain of dependent steps. A thread keeps four columns of
// DR rows of HP heads' states in registers, asked for before anything else. With a = g S (decayed rows) one pass gives both
// a^T k and a^T q, and as S' = a + k u^T reads out as a^T q + u (k.q), the sums over rows cross the waves once a step. All
// loads that wait for nothing go out together, and 128 registers hold two workgroups on a compute unit. In place of eight
// launches; 16 heads of 64 x 128 on 8 key heads: 8 rows 12 us, 40 rows 18.5 (24.4 with 145 registers; the state alone
// takes 9 at the rate of a copy); a step of 8 rows 586 us before, 444 with it, of 40 rows 679 and 564.
struct DeltaColumns { int at[6]; };

#define DR_THREADS 512
#define DR_OUTS 6             // low-rank outputs of eight lanes at a time: registers
#define DR_BLOCK 128           // columns of the state at a time

template <int DR, int HP, int TAPS>
__global__ void __launch_bounds__(DR_THREADS, DR * HP <= 8 ? 4 : 2) delta_rows_kernel(
    const float* __restrict__ part, int S, DeltaColumns cols, const float* __restrict__ conv, bfraw* __restrict__ conv_state,
    int K, int C, const bfraw* __restrict__ a2, int RA, const bfraw* __restrict__ g2, int RB,
    const float* __restrict__ dt_bias, const float* __restrict__ a_log, float* __restrict__ state,
    const float* __restrict__ norm, bfraw* __restrict__ out, const int* __restrict__ slots, const int* __restrict__ cu,
    const int* __restrict__ seg_start, int T_, int N, int H, int G, int D, int V, float eps) {
  extern __shared__ float lds[];
  const int b = blockIdx.y, g = blockIdx.x, tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
  const int rep = H / G, h0 = g * rep;
  float* const ks = lds, *const qs = ks + D, *const vs = qs + D;
  bfraw* const low = reinterpret_cast<bfraw*>(lds + (2 * D + rep * V + 3) / 4 * 4);   // RA and RB are multiples of 8
  float* const us = reinterpret_cast<float*>(low + RA + RB), *const red = us + HP * DR_BLOCK, *const dec = red + HP * 2 * DR_THREADS * 4;
  float* const gate = dec + rep * D, *const nw = gate + rep * V, *const beta = nw + V, *const kq = beta + rep;
  const int t = cu[b];
  if (cu[b + 1] == t) return;                         // the whole workgroup
  const bool fresh = seg_start[b] == 0;
  const int64_t slot = slots[b];
  f32x4 st[HP][DR];
  auto fetch = [&](int hh, int c0, int V4, int RG) {
    const int quad = tid % V4, rg = tid / V4;
#pragma unroll
    for (int p = 0; p < HP; ++p) {
      const float* sp = state + ((slot * H + h0 + hh + p) * D) * (int64_t)V + c0 + quad * 4;
#pragma unroll
      for (int i = 0; i < DR; ++i) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(sp + (int64_t)min(i * RG + rg, D - 1) * V);
        st[p][i] = fresh ? f32x4{0.f, 0.f, 0.f, 0.f} : v;
      }
    }
  };

  // the columns this workgroup reads: k, q, v (convolved), the two low-rank inputs, and beside them the write strengths;
  // the loads of a thread's column by themselves, eight shares and, of the unused taps, the last ones' places
  const int conv_n = 2 * D + rep * V, low_n = conv_n + RA + RB, plane = T_ * N;
  float v[8], e[8], tap[TAPS], norm_w;
  bfraw old[TAPS - 1], *hist;
  int to_beta;
  const float* p;
  auto column = [&](int i) {
    int c = cols.at[1];
    if (i < D) c = cols.at[1] + g * D + i;
    else if (i < 2 * D) c = cols.at[0] + g * D + i - D;
    else if (i < conv_n) c = cols.at[2] + h0 * V + i - 2 * D;
    const int ch = c;
    if (i >= conv_n && i < conv_n + RA) c = cols.at[3] + i - conv_n;
    else if (i >= conv_n && i < low_n) c = cols.at[4] + i - conv_n - RA;
    p = part + (int64_t)t * N + c;
    to_beta = i < rep ? cols.at[5] + h0 + i - c : 0;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      v[s] = p[(int64_t)min(s, S - 1) * plane];
      e[s] = p[(int64_t)min(s, S - 1) * plane + to_beta];
    }
    hist = conv_state + slot * (K - 1) * C + ch;
#pragma unroll
    for (int j = 0; j < TAPS - 1; ++j) {
      old[j] = hist[(int64_t)min(j, K - 2) * C];
      tap[j] = conv[(int64_t)min(j, K - 1) * C + ch];
    }
    tap[TAPS - 1] = conv[(int64_t)(K - 1) * C + ch];
    norm_w = norm[min(i, V - 1)];
  };
  column(tid);

  // first weights of the low-rank products: eight lanes an output, output u of DR_OUTS at tid / 8 + 64 u
  const int sub = lane % 8, outs = rep * (D + V);
  uint4 w[DR_OUTS];
  auto weights = [&](int o0, int r) {
#pragma unroll
    for (int u = 0; u < DR_OUTS; ++u) {
      const int o = min(o0 + 64 * u, outs - 1);
      const bool is_a = o < rep * D;
      w[u] = *reinterpret_cast<const uint4*>(is_a ? a2 + (int64_t)(h0 * D + o) * RA + min(r, RA - 8)
                                                  : g2 + (int64_t)(h0 * V + o - rep * D) * RB + min(r, RB - 8));
    }
  };
  const int mine = min(tid / 8 + 64 * sub, rep * D - 1);
  const float dt0 = dt_bias[h0 * D + mine], log0 = a_log[h0 + mine / D];
  {
    const int V4 = min(V, DR_BLOCK) / 4;
    fetch(0, 0, V4, DR_THREADS / V4);
  }
  for (int i = tid; i < max(low_n, V); i += DR_THREADS) {
    if (i >= DR_THREADS) column(i);
    float x = 0.0f, strength = 0.0f;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      x += s < S ? v[s] : 0.0f;
      strength += s < S ? e[s] : 0.0f;
    }
    for (int s = 8; s < S; ++s) {
      x += p[(int64_t)s * plane];
      strength += p[(int64_t)s * plane + to_beta];
    }
    const uint32_t bits = bf_bits(x);
    x = __uint_as_float(bits << 16);
    if (i < rep) beta[i] = sigmoid_exact(__uint_as_float(bf_bits(strength) << 16));
    if (i < V) nw[i] = norm_w;
    if (i < conv_n) {
      float acc = 0.0f;
#pragma unroll
      for (int j = 0; j < TAPS - 1; ++j) {
        if (fresh) old[j] = 0;
        if (j < K - 1 && !fresh) acc += tap[j] * ldf(old + j);
      }
      acc += tap[TAPS - 1] * x;
#pragma unroll
      for (int j = 1; j < TAPS - 1; ++j)
        if (j < K - 1) hist[(int64_t)(j - 1) * C] = old[j];
      hist[(int64_t)(K - 2) * C] = (bfraw)bits;
      lds[i] = __uint_as_float(bf_bits(silu_exact(acc)) << 16);
    } else if (i < low_n) {
      low[i - conv_n] = (bfraw)bits;
    }
  }
  weights(tid / 8, sub * 8);
  __syncthreads();

  // in the first wave the unit k and q; then the low-rank products, of which each of the first lanes of eight finishes one
  if (wave == 0) {
    float sk = 0.0f, sq = 0.0f, d2 = 0.0f;
    for (int d = lane; d < D; d += WAVE) { sk += ks[d] * ks[d]; sq += qs[d] * qs[d]; d2 += ks[d] * qs[d]; }
    sk = group_sum<1>(sk);
    sq = group_sum<1>(sq);
    d2 = group_sum<1>(d2);
    const float rq = 1.0f / (sqrtf(sq + 1e-6f) * sqrtf((float)D)), rk = 1.0f / sqrtf(sk + 1e-6f);
    for (int d = lane; d < D; d += WAVE) { ks[d] *= rk; qs[d] *= rq; }
    if (lane == 0) *kq = d2 * rq * rk;
  }
  for (int o0 = tid / 8; o0 - tid / 8 < outs; o0 += 64 * DR_OUTS) {
    const bool first = o0 < 64 * DR_OUTS;
    float acc[DR_OUTS] = {}, sum = 0.0f;
    for (int r0 = 0; r0 < max(RA, RB); r0 += 64) {
      const int r = r0 + sub * 8;
      if (!first || r0 > 0) weights(o0, r);
      const uint4 xa = *reinterpret_cast<const uint4*>(low + min(r, RA - 8));
      const uint4 xb = *reinterpret_cast<const uint4*>(low + RA + min(r, RB - 8));
#pragma unroll
      for (int u = 0; u < DR_OUTS; ++u) {
        const bool is_a = o0 + 64 * u < rep * D;
        const int R = is_a ? RA : RB;
        const uint32_t ws[4] = {w[u].x, w[u].y, w[u].z, w[u].w};
        const uint32_t xs[4] = {is_a ? xa.x : xb.x, is_a ? xa.y : xb.y, is_a ? xa.z : xb.z, is_a ? xa.w : xb.w};
        float more = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; ++k)
          more += __uint_as_float(ws[k] << 16) * __uint_as_float(xs[k] << 16) +
                  __uint_as_float(ws[k] & 0xffff0000u) * __uint_as_float(xs[k] & 0xffff0000u);
        acc[u] += r < R ? more : 0.0f;
      }
    }
#pragma unroll
    for (int off = 1; off < 8; off <<= 1)
#pragma unroll
      for (int u = 0; u < DR_OUTS; ++u) acc[u] += __shfl_xor(acc[u], off);
#pragma unroll
    for (int u = 0; u < DR_OUTS; ++u) sum = u == sub ? acc[u] : sum;
    const int o = o0 + 64 * sub;
    if (sub >= DR_OUTS || o >= outs) continue;
    sum = __uint_as_float(bf_bits(sum) << 16);
    if (o < rep * D)
      dec[o] = expf(-expf(first ? log0 : a_log[h0 + o / D]) * softplus_exact(sum + (first ? dt0 : dt_bias[h0 * D + o])));
    else
      gate[o - rep * D] = sigmoid_exact(sum);
  }
  __syncthreads();

  for (int hh = 0; hh < rep; hh += HP) {
    for (int c0 = 0; c0 < V; c0 += DR_BLOCK) {
      const int VB = min(V - c0, DR_BLOCK), V4 = VB / 4, RG = DR_THREADS / V4, quad = tid % V4, rg = tid / V4;
      if (hh + c0 > 0) fetch(hh, c0, V4, RG);
#pragma unroll
      for (int p = 0; p < HP; ++p) {
        f32x4 pred = {0.f, 0.f, 0.f, 0.f}, read = pred;
#pragma unroll
        for (int i = 0; i < DR; ++i) {
          const int d = min(i * RG + rg, D - 1);
          const bool on = i * RG + rg < D;
          const float dc = dec[(hh + p) * D + d], k = on ? ks[d] : 0.0f, q = on ? qs[d] : 0.0f;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            st[p][i][e] *= dc;
            pred[e] += st[p][i][e] * k;
            read[e] += st[p][i][e] * q;
          }
        }
        if (rg < RG) {
          *reinterpret_cast<f32x4*>(red + (p * 2 * RG + rg) * VB + quad * 4) = pred;
          *reinterpret_cast<f32x4*>(red + ((p * 2 + 1) * RG + rg) * VB + quad * 4) = read;
        }
      }
      __syncthreads();
      if (tid < HP * VB) {
        const int p = tid / VB, c = tid % VB;
        const float* r = red + p * 2 * RG * VB + c;
        float pred = 0.0f, read = 0.0f;
#pragma unroll 8
        for (int i = 0; i < RG; ++i) { pred += r[i * VB]; read += r[(RG + i) * VB]; }
        float* val = vs + (hh + p) * V + c0 + c;
        const float u = beta[hh + p] * (*val - pred);
        us[p * DR_BLOCK + c] = u;
        *val = read + u * *kq;
      }
      __syncthreads();
#pragma unroll
      for (int p = 0; p < HP; ++p) {
        float* sp = state + ((slot * H + h0 + hh + p) * D) * (int64_t)V + c0 + quad * 4;
        const f32x4 u = *reinterpret_cast<const f32x4*>(us + p * DR_BLOCK + quad * 4);
#pragma unroll
        for (int i = 0; i < DR; ++i) {
          const int d = i * RG + rg;
          if (d >= D || rg >= RG) continue;
          const float k = ks[d];
#pragma unroll
          for (int e = 0; e < 4; ++e) st[p][i][e] += k * u[e];
          *reinterpret_cast<f32x4*>(sp + (int64_t)d * V) = st[p][i];
        }
      }
    }
  }
  for (int p = wave; p < rep; p += DR_THREADS / WAVE) {
    const float* o = vs + p * V;
    float ss = 0.0f;
    for (int c = lane; c < V; c += WAVE) ss += o[c] * o[c];
    const float r = 1.0f / sqrtf(group_sum<1>(ss) / (float)V + eps);
    for (int c = lane; c < V; c += WAVE) stf(out + ((int64_t)t * H + h0 + p) * V + c, o[c] * r * nw[c] * gate[p * V + c]);
  }
}

static inline size_t delta_rows_lds(int rep, int D, int V, int ranks, int HP) {
  return ((size_t)2 * D + rep * (2 * V + D + 1) + V + ranks + 1 + 3 + HP * (DR_BLOCK + 2 * DR_THREADS * 4)) * sizeof(float);
}

// false, and nothing done, for sizes it is not written for: value sizes and ranks in fours and eights, keys up to 256, what
// a workgroup keeps within 64 KB
extern "C" bool seq_delta_rows_takes(int H, int G, int D, int V, int K, int RA, int RB) {
  const int rep = H / G;
  return D <= 256 && V % 4 == 0 && K >= 2 && K <= 16 && RA % 8 == 0 && RB % 8 == 0 &&
         delta_rows_lds(rep, D, V, RA + RB, rep % 2 == 0 ? 2 : 1) <= 65536;
}

extern "C" void seq_launch_delta_rows(const float* part, int S, const int64_t* at, const float* conv, void* conv_state, int K,
                                      int C, const void* a2, int RA, const void* g2, int RB, const float* dt_bias,
                                      const float* a_log, float* state, const float* norm, void* out, const int* slots,
                                      const int* cu, const int* seg_start, int T_, int N, int H, int G, int D, int V,
                                      float eps, hipStream_t st) {
  DeltaColumns cols;
  for (int i = 0; i < 6; ++i) cols.at[i] = (int)at[i];
  const int rep = H / G, RG = DR_THREADS / ((V < DR_BLOCK ? V : DR_BLOCK) / 4), rows = (D + RG - 1) / RG;
  auto go = [&](auto kernel, int HP) {
    hipLaunchKernelGGL(kernel, dim3(G, T_), dim3(DR_THREADS), delta_rows_lds(rep, D, V, RA + RB, HP), st, part, S, cols, conv,
                       (bfraw*)conv_state, K, C, (const bfraw*)a2, RA, (const bfraw*)g2, RB, dt_bias, a_log, state, norm,
                       (bfraw*)out, slots, cu, seg_start, T_, N, H, G, D, V, eps);
  };
  auto by_taps = [&](auto few, auto many, int HP) { K <= 4 ? go(few, HP) : go(many, HP); };
  const bool two = rep % 2 == 0;
  if (rows <= 4 && two) by_taps(delta_rows_kernel<4, 2, 4>, delta_rows_kernel<4, 2, 16>, 2);
  else if (rows <= 4) by_taps(delta_rows_kernel<4, 1, 4>, delta_rows_kernel<4, 1, 16>, 1);
  else if (rows <= 8 && two) by_taps(delta_rows_kernel<8, 2, 4>, delta_rows_kernel<8, 2, 16>, 2);
  else if (rows <= 8) by_taps(delta_rows_kernel<8, 1, 4>, delta_rows_kernel<8, 1, 16>, 1);
  else by_taps(delta_rows_kernel<16, 1, 4>, delta_rows_kernel<16, 1, 16>, 1);
}
