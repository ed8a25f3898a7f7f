// Row-wise passes of a hybrid model's step of few rows, straight from the split sums of the product before them
// (fp32, as linear_rows leaves them). First the residual epilogue, a [SA, T, W], b [SB, T, W]:
//   y = a, or (rms(a) wa + rms(b / rms(what b is of)) wb) / 2;  x += rms(y) w_post;  out = rms(x) w_next in bf16
//
// A row is one workgroup's: its sums are the bytes, 64 to 128 KB of them, and the three reductions the chain behind. Four
// columns a thread and load, kept in registers through all passes, and all loads before the first wait. 40 rows of 2048 in 8
// shares: 3.9 us of a step, with two branches of 4 shares 4.8 (4.7 and 8.3 with the loads one by one behind the shares that
// fill a batch, and three of the norms' weights behind the sums).

#include "seq_common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define SR_THREADS 512

// Sums of S splits a plane apart, in their order; the loads of four or eight go out together, those past the last one to its
// place
__device__ __forceinline__ f32x4 split_sum(const float* __restrict__ p, int S, int64_t plane) {
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
  if (S <= 4) {
    f32x4 v[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) v[s] = *reinterpret_cast<const f32x4*>(p + min(s, S - 1) * plane);
#pragma unroll
    for (int s = 0; s < 4; ++s)
      if (s < S) sum += v[s];
    return sum;
  }
  for (int s0 = 0; s0 < S; s0 += 8) {
    f32x4 v[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) v[s] = *reinterpret_cast<const f32x4*>(p + min(s0 + s, S - 1) * plane);
#pragma unroll
    for (int s = 0; s < 8; ++s)
      if (s0 + s < S) sum += v[s];
  }
  return sum;
}

// VECS: W <= 4 * VECS * SR_THREADS
template <bool DUAL, int VECS>
__global__ void __launch_bounds__(SR_THREADS) sandwich_rows_kernel(
    float* __restrict__ x, const float* __restrict__ a, int SA, const float* __restrict__ b, int SB,
    const float* __restrict__ wa, const float* __restrict__ wb, const float* __restrict__ w_post,
    const float* __restrict__ w_next, bfraw* __restrict__ out, int T_, int W, float eps,
    const float* __restrict__ squares, int heads, float per) {
  __shared__ float scratch[2][16];
  const int t = blockIdx.x, tid = threadIdx.x, nvec = W / 4;
  const int64_t plane = (int64_t)T_ * W;
  const float inv_w = 1.0f / (float)W;
  f32x4 y[VECS], z[VECS], old[VECS], post[VECS], next[VECS], ga[VECS], gb[VECS];
  float ss = 0.0f, sb = 0.0f, sq = 0.0f;
  // b is of a product whose rows' norm is put off to here
  if constexpr (DUAL)
    for (int i = tid % WAVE; i < heads; i += WAVE) sq += squares[(int64_t)t * heads + i];
#pragma unroll
  for (int k = 0; k < VECS; ++k) {
    const int i = tid + k * SR_THREADS;
    if (i >= nvec) break;
    const int64_t at = (int64_t)t * W + i * 4;
    old[k] = *reinterpret_cast<const f32x4*>(x + at);
    post[k] = reinterpret_cast<const f32x4*>(w_post)[i];
    next[k] = reinterpret_cast<const f32x4*>(w_next)[i];
    if constexpr (DUAL) {
      ga[k] = reinterpret_cast<const f32x4*>(wa)[i];
      gb[k] = reinterpret_cast<const f32x4*>(wb)[i];
      z[k] = split_sum(b + at, SB, plane);
#pragma unroll
      for (int e = 0; e < 4; ++e) sb += z[k][e] * z[k][e];
    }
    y[k] = split_sum(a + at, SA, plane);
#pragma unroll
    for (int e = 0; e < 4; ++e) ss += y[k][e] * y[k][e];
  }
  if constexpr (DUAL) {
    const float rs = 1.0f / sqrtf(group_sum<1>(sq) * per + eps);
    // both sums over the row behind one barrier
    const int lane = tid % WAVE, wave = tid / WAVE;
    ss = group_sum<1>(ss);
    sb = group_sum<1>(sb * rs * rs);
    if (lane == 0) { scratch[0][wave] = ss; scratch[1][wave] = sb; }
    __syncthreads();
    ss = sb = 0.0f;
#pragma unroll
    for (int i = 0; i < SR_THREADS / WAVE; ++i) { ss += scratch[0][i]; sb += scratch[1][i]; }
    const float ra = 1.0f / sqrtf(ss * inv_w + eps), rb = 1.0f / sqrtf(sb * inv_w + eps);
    ss = 0.0f;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < VECS; ++k) {
      if (tid + k * SR_THREADS >= nvec) break;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        y[k][e] = 0.5f * (y[k][e] * ra * ga[k][e] + z[k][e] * rs * rb * gb[k][e]);
        ss += y[k][e] * y[k][e];
      }
    }
  }
  // two sums, one behind the other, each in a place of its own
  auto row_sum = [&](float v, float* place) {
    v = group_sum<1>(v);
    if (tid % WAVE == 0) place[tid / WAVE] = v;
    __syncthreads();
    v = 0.0f;
#pragma unroll
    for (int i = 0; i < SR_THREADS / WAVE; ++i) v += place[i];
    return v;
  };
  const float ry = 1.0f / sqrtf(row_sum(ss, scratch[0]) * inv_w + eps);
  float sx = 0.0f;
#pragma unroll
  for (int k = 0; k < VECS; ++k) {
    const int i = tid + k * SR_THREADS;
    if (i >= nvec) break;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      y[k][e] = old[k][e] + y[k][e] * ry * post[k][e];
      sx += y[k][e] * y[k][e];
    }
    reinterpret_cast<f32x4*>(x + (int64_t)t * W)[i] = y[k];
  }
  const float rx = 1.0f / sqrtf(row_sum(sx, scratch[1]) * inv_w + eps);
#pragma unroll
  for (int k = 0; k < VECS; ++k) {
    const int i = tid + k * SR_THREADS;
    if (i >= nvec) break;
    uint2 o;
    o.x = bf_bits(y[k][0] * rx * next[k][0]) | (bf_bits(y[k][1] * rx * next[k][1]) << 16);
    o.y = bf_bits(y[k][2] * rx * next[k][2]) | (bf_bits(y[k][3] * rx * next[k][3]) << 16);
    reinterpret_cast<uint2*>(out + (int64_t)t * W)[i] = o;
  }
}

// b nullptr: one branch. squares [T, heads]: sums of squares of which per times the row's total is the mean that b's rows are
// still to be normalised by
extern "C" void seq_launch_sandwich_rows(float* x, const float* a, int SA, const float* b, int SB, const float* wa,
                                         const float* wb, const float* w_post, const float* w_next, void* out, int T_,
                                         int W, float eps, const float* squares, int heads, float per, hipStream_t st) {
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(T_), dim3(SR_THREADS), 0, st, x, a, SA, b, SB, wa, wb, w_post, w_next, (bfraw*)out, T_, W,
                       eps, squares, heads, per);
  };
  const bool narrow = W <= 4 * SR_THREADS;
  if (b) narrow ? go(sandwich_rows_kernel<true, 1>) : go(sandwich_rows_kernel<true, 4>);
  else narrow ? go(sandwich_rows_kernel<false, 1>) : go(sandwich_rows_kernel<false, 4>);
}

// What a parallel sublayer's input product, as split sums part [S, T, N], is wanted for, in one launch: sums (+ bias), then for
// the softmax branch left q rotated in pairs and rounded, left k rotated into the cache with itself as the value and the head
// gates rounded (four columns a thread); and the recurrent branch up to its norm, a workgroup a row's head: silu of q, k, v,
// the step of the recurrence, and o w sigmoid(gate) in bf16 with the head's sum of o^2, from which the branch's norm over all
// heads is one factor a row for the pass behind the output product. at: first columns of left q, k, head gates and right q, k,
// v, gate, all multiples of 8.
//
// Bound by the state's bytes (32 KB a head of 64 x 128, read and written). A thread keeps four columns of DR rows of the state.
// In place of a pass over the sums, the recurrence and the norm (4.5, 14.5 and 5 us for 40 rows of 16 heads): 12.9 us, with 8
// rows 6.8 (15).
struct SplitColumns { int at[7]; };

#define PR_THREADS 512
#define DR_BLOCK 128           // columns of the state at a time

template <int DR>
__global__ void __launch_bounds__(PR_THREADS, DR <= 8 ? 4 : 2) parallel_rows_kernel(
    const float* __restrict__ part, int S, const bfraw* __restrict__ bias, SplitColumns cols,
    const int64_t* __restrict__ positions, const float* __restrict__ inv_freq, bfraw* __restrict__ k_cache,
    bfraw* __restrict__ v_cache, const int64_t* __restrict__ cache_slots, bfraw* __restrict__ q_out,
    bfraw* __restrict__ head_gate, const float* __restrict__ decay, float* __restrict__ state,
    const float* __restrict__ norm, bfraw* __restrict__ z, float* __restrict__ squares,
    const int* __restrict__ slots, const int* __restrict__ cu, const int* __restrict__ seg_start, int T_, int N, int H,
    int G, int R, int BS, int RH, int RD, int RV) {
  extern __shared__ float lds[];
  const int tid = threadIdx.x, plane = T_ * N;
  if ((int)blockIdx.x >= RH) {
    const int t = blockIdx.y, i = ((blockIdx.x - RH) * PR_THREADS + tid) * 4;
    const int nq = H * 128, nk = G * 128;
    if (i >= nq + nk + H) return;
    const bool is_q = i < nq, is_k = !is_q && i < nq + nk;
    const int o = is_q ? i : is_k ? i - nq : i - nq - nk, c = cols.at[is_q ? 0 : is_k ? 1 : 2] + o;
    const float* p = part + (int64_t)t * N + c;
    float x[4] = {};
    for (int s0 = 0; s0 < S; s0 += 8) {
      f32x4 v[8];
#pragma unroll
      for (int s = 0; s < 8; ++s) v[s] = *reinterpret_cast<const f32x4*>(p + (int64_t)min(s0 + s, S - 1) * plane);
#pragma unroll
      for (int s = 0; s < 8; ++s)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] += s0 + s < S ? v[s][e] : 0.0f;
    }
    if (bias) {
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] += ldf(bias + c + e);
    }
    auto put = [](bfraw* to, const float (&v)[4]) {
      *reinterpret_cast<uint2*>(to) = make_uint2(bf_bits(v[0]) | (bf_bits(v[1]) << 16), bf_bits(v[2]) | (bf_bits(v[3]) << 16));
    };
    if (!is_q && !is_k) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (o + e < H) stf(head_gate + (int64_t)t * H + o + e, x[e]);
      return;
    }
    const int dim = o % 128;
    float y[4];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      float sn = 0.0f, cs = 1.0f;
      if (dim / 2 + k < R) sincosf((float)positions[t] * inv_freq[dim / 2 + k], &sn, &cs);
      y[2 * k] = x[2 * k] * cs - x[2 * k + 1] * sn;
      y[2 * k + 1] = x[2 * k + 1] * cs + x[2 * k] * sn;
    }
    if (is_q) {
      put(q_out + (int64_t)t * nq + o, y);
    } else {
      const int64_t slot = cache_slots[t], row = (slot / BS * G + o / 128) * BS + slot % BS;
      put(k_cache + row * 128 + dim, y);
      put(v_cache + row * 128 + dim, x);
    }
    return;
  }
  const int b = blockIdx.y, h = blockIdx.x, t = cu[b];
  if (cu[b + 1] == t) return;                         // the whole workgroup
  const bool fresh = seg_start[b] == 0;
  float* const qs = lds, *const ks = qs + RD, *const vs = ks + RD, *const gate = vs + RV;
  float* const red = gate + RV;                       // RD and RV are multiples of 4
  const float dec = decay[h];
  float* const head = state + ((int64_t)slots[b] * RH + h) * RD * RV;
  f32x4 st[DR];
  auto fetch = [&](int c0, int V4, int RG) {
    const int quad = tid % V4, rg = tid / V4;
#pragma unroll
    for (int i = 0; i < DR; ++i) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(head + (int64_t)min(i * RG + rg, RD - 1) * RV + c0 + quad * 4);
      st[i] = fresh ? f32x4{0.f, 0.f, 0.f, 0.f} : v;
    }
  };
  const int n = 2 * (RD + RV);
  float v[8], add = 0.0f;
  const float* p;
  auto column = [&](int i) {
    i = min(i, n - 1);
    const int c = i < RD ? cols.at[3] + h * RD + i : i < 2 * RD ? cols.at[4] + h * RD + i - RD
                : i < 2 * RD + RV ? cols.at[5] + h * RV + i - 2 * RD : cols.at[6] + h * RV + i - 2 * RD - RV;
    p = part + (int64_t)t * N + c;
#pragma unroll
    for (int s = 0; s < 8; ++s) v[s] = p[(int64_t)min(s, S - 1) * plane];
    if (bias) add = ldf(bias + c);
  };
  column(tid);
  const int first4 = min(RV, DR_BLOCK) / 4;
  fetch(0, first4, PR_THREADS / first4);
  for (int i = tid; i < n; i += PR_THREADS) {
    if (i >= PR_THREADS) column(i);
    float x = 0.0f;
#pragma unroll
    for (int s = 0; s < 8; ++s) x += s < S ? v[s] : 0.0f;
    for (int s = 8; s < S; ++s) x += p[(int64_t)s * plane];
    x += add;
    lds[i] = i < 2 * RD + RV ? silu_exact(x) : sigmoid_exact(__uint_as_float(bf_bits(x) << 16));
  }
  __syncthreads();
  float ss = 0.0f;
  for (int c0 = 0; c0 < RV; c0 += DR_BLOCK) {
    const int VB = min(RV - c0, DR_BLOCK), V4 = VB / 4, RG = PR_THREADS / V4, quad = tid % V4, rg = tid / V4;
    if (c0 > 0) fetch(c0, V4, RG);
    f32x4 read = {0.f, 0.f, 0.f, 0.f};
    if (rg < RG) {
      const f32x4 val = *reinterpret_cast<const f32x4*>(vs + c0 + quad * 4);
#pragma unroll
      for (int i = 0; i < DR; ++i) {
        const int d = i * RG + rg;
        const bool on = d < RD;
        const float k = ks[min(d, RD - 1)], q = on ? qs[min(d, RD - 1)] : 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          st[i][e] = on ? dec * st[i][e] + k * val[e] : 0.0f;
          read[e] += st[i][e] * q;
        }
        if (on) *reinterpret_cast<f32x4*>(head + (int64_t)d * RV + c0 + quad * 4) = st[i];
      }
      *reinterpret_cast<f32x4*>(red + rg * VB + quad * 4) = read;
    }
    __syncthreads();
    if (tid < VB) {
      float o = 0.0f;
#pragma unroll 8
      for (int i = 0; i < RG; ++i) o += red[i * VB + tid];
      ss += o * o;
      const int c = c0 + tid;
      stf(z + ((int64_t)t * RH + h) * RV + c, o * norm[h * RV + c] * gate[c]);
    }
    __syncthreads();
  }
  ss = block_sum(ss, red);
  if (tid == 0) squares[(int64_t)t * RH + h] = ss;
}

static inline size_t parallel_rows_lds(int RD, int RV) { return (size_t)(2 * (RD + RV) + PR_THREADS * 4) * sizeof(float); }

// what a workgroup keeps within 64 KB
extern "C" bool seq_parallel_rows_takes(int RD, int RV) { return RD <= 256 && parallel_rows_lds(RD, RV) <= 65536; }

extern "C" void seq_launch_parallel_rows(const float* part, int S, const void* bias, const int64_t* at,
                                         const int64_t* positions, const float* inv_freq, void* k_cache, void* v_cache,
                                         const int64_t* cache_slots, void* q_out, void* head_gate, const float* decay,
                                         float* state, const float* norm, void* z, float* squares,
                                         const int* slots, const int* cu, const int* seg_start, int T_, int N, int H, int G,
                                         int R, int BS, int RH, int RD, int RV, hipStream_t st) {
  SplitColumns cols;
  for (int i = 0; i < 7; ++i) cols.at[i] = (int)at[i];
  const int left = (H * 128 + G * 128 + H + 4 * PR_THREADS - 1) / (4 * PR_THREADS);
  const int RG = PR_THREADS / ((RV < DR_BLOCK ? RV : DR_BLOCK) / 4), rows = (RD + RG - 1) / RG;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(RH + left, T_), dim3(PR_THREADS), parallel_rows_lds(RD, RV), st, part, S,
                       (const bfraw*)bias, cols, positions, inv_freq, (bfraw*)k_cache, (bfraw*)v_cache, cache_slots,
                       (bfraw*)q_out, (bfraw*)head_gate, decay, state, norm, (bfraw*)z, squares, slots, cu,
                       seg_start, T_, N, H, G, R, BS, RH, RD, RV);
  };
  if (rows <= 4) go(parallel_rows_kernel<4>);
  else if (rows <= 8) go(parallel_rows_kernel<8>);
  else go(parallel_rows_kernel<16>);
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
            st[p][i][e] = on ? st[p][i][e] * dc : 0.0f;
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

// false for sizes it is not written for: value sizes and ranks in fours and eights, keys up to 256, what
// a workgroup keeps within 64 KB
extern "C" bool seq_delta_rows_takes(int H, int G, int D, int V, int K, int RA, int RB) {
  const int rep = H / G;
  return D <= 256 && V % 4 == 0 && K >= 2 && K <= 16 && RA >= 8 && RA % 8 == 0 && RB >= 8 && RB % 8 == 0 &&
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
