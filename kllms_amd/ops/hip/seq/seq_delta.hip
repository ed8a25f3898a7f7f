// The gated delta rule over prompts, 16 tokens at a time, for key size 64 (gfx950).
//
//   S <- g_t (.) S;  u_t = beta_t (v_t - S^T k_t);  S <- S + k_t u_t^T;  o_t = S^T q_t
//
// Token by token a head's chain of two reductions a token is the bound: 0.46 us each, whatever the chip has idle. Over
// a chunk of 16 tokens, with S0 the state before it and P_ts the product of g over (s, t] (P_t from the chunk's start),
//
//   (I + L) U = beta (V - (P k) S0),   L_ts = beta_t sum_d k_t k_s P_ts (s < t)
//   O = (P q) S0 + M U,                M_ts = sum_d q_t k_s P_ts (s <= t)
//   S = P_16 S0 + sum_s (P_16s k_s) u_s^T
//
// so that only the products with S0 and U are left in the chain. All else is of the chunk alone:
//
//   delta_chunk   a wave per (chunk, head): L and M, the inverse T of I + L by substitution, T beta (P k) and T beta V
//   delta_scan    a wave per (segment, head, 16 value columns): chunk after chunk, 52 matrix instructions each
//
// The matrix instructions add up all 16 tokens, with a zero in L, T or M for those to come, and zero times infinity is
// NaN: from a token on whose k, write strength or decay is not finite, and in a column from a v on that is not, operands
// are zeros, and the rows become NaN. So nothing reaches an earlier token, as token by token.
//
// Everything stays in fp32 (v_mfma_f32_16x16x4_f32), and no decay is divided by or taken as an exponential of a
// difference: the P are running products of factors in (0, 1], as token by token. The state's registers are both
// the B operand of the products and the accumulators of the update: k runs in the order d = 16 m + 4 grp + r.
//
// What bounds them: delta_chunk its records (21 KB a chunk and head: 166 MB in 142 us for 8 x 1000 tokens, 16 heads) and
// the pairs' sums, delta_scan its matrix instructions, 1700 cycles a chunk, with one wave on a SIMD and two chunks of
// operands on their way (128 us; 150 with one). Together, us, beside token by token with its pre-pass, 16 heads of 64 x 128:
// 1 x 100 tokens 40 (47), 1 x 1000 124 (394), 8 x 1000 262 (547), 4 x 2000 333 (850), 64 x 250 of 32 heads of 64 x 64 714 (1158).

#include "seq_common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define DC_C 16                          // tokens of a chunk
#define DC_D 64                          // key size
// record of a (chunk, head): W [16][64], Q [16][64], Kt [64][16], M [16][16], P [64], U [16][V]
#define DC_W 0
#define DC_Q 1024
#define DC_K 2048
#define DC_M 3072
#define DC_P 3328
#define DC_U 3392

// chunks of segment b begin at slot cu[b] / 16 + b: no two segments' overlap, T / 16 + B slots hold all
__device__ __forceinline__ int chunk_base(const int* cu, int b) { return cu[b] / DC_C + b; }

__device__ __forceinline__ float row_sum16(float v) {   // over 16 lanes, every lane gets it
  v += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0x128, 0xf, 0xf, false));   // row_ror 8, 4, 2, 1
  v += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0x124, 0xf, 0xf, false));
  v += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0x122, 0xf, 0xf, false));
  v += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0x121, 0xf, 0xf, false));
  return v;
}

// Not 0 where one of the values is infinite or NaN (no comparison that could be taken for granted: x - x is 0 or NaN)
__device__ __forceinline__ float not_finite(const f32x4& v) {
  return (v[0] - v[0]) + (v[1] - v[1]) + ((v[2] - v[2]) + (v[3] - v[3]));
}

// Rows of a result in matrix layout (row 4 grp + r, column col): the first one of each column whose value is not finite, 16: none
__device__ __forceinline__ int first_odd_row(const f32x4& v, int col) {
  int first = 16;
#pragma unroll
  for (int r = 3; r >= 0; --r) {
    const unsigned long long odd = __ballot(v[r] - v[r] != 0.0f) >> col;
#pragma unroll
    for (int g = 3; g >= 0; --g)
      if ((odd >> (g * 16)) & 1) first = min(first, g * 4 + r);
  }
  return first;
}

template <typename T>
__global__ void __launch_bounds__(WAVE) delta_chunk_kernel(
    float* __restrict__ rec, const T* __restrict__ q_in, const T* __restrict__ k_in, const T* __restrict__ v_in,
    const T* __restrict__ beta_logit, const T* __restrict__ a_in, const float* __restrict__ dt_bias,
    const float* __restrict__ a_log, const int* __restrict__ cu, int B, int H, int G, int V, int q_stride, int k_stride,
    int v_stride, int beta_stride, int a_stride) {
  __shared__ __attribute__((aligned(16))) float k[DC_C][DC_D], q[DC_C][DC_D], g[DC_C][DC_D];
  __shared__ float L[DC_C][DC_C + 1], M[DC_C][DC_C + 1], Ti[DC_C][DC_C + 1], beta[DC_C];
  const int lane = threadIdx.x, col = lane & 15, grp = lane >> 4;
  const int slot = blockIdx.x, h = blockIdx.y, kv = h / (H / G);
  int b = -1;
  for (int c = 0; c < B && b < 0; c += WAVE) {
    const int i = c + lane;
    const bool in = i < B && slot >= chunk_base(cu, i) && slot < chunk_base(cu, i) + (cu[i + 1] - cu[i] + DC_C - 1) / DC_C;
    const unsigned long long any = __ballot(in);
    if (any) b = c + __builtin_ctzll(any);
  }
  if (b < 0) return;
  const int t0 = cu[b] + (slot - chunk_base(cu, b)) * DC_C, n = min(DC_C, cu[b + 1] - t0);
  float* r0 = rec + ((int64_t)slot * H + h) * (DC_U + DC_C * V);

  // unit q and k, q by 1 / sqrt(64), decays and write strengths; behind the segment's end k, q and beta 0, decay 1
  const float rate = expf(a_log[h]);
  int bad = DC_C;                          // first token with a k, decay or write strength that is not finite
  f32x4 dt;
#pragma unroll
  for (int x = 0; x < 4; ++x) dt[x] = dt_bias[h * DC_D + col * 4 + x];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = i * 4 + grp;
    const int64_t row = t0 + min(t, n - 1);
    const T *pk = k_in + row * k_stride + kv * DC_D + col * 4, *pq = q_in + row * q_stride + kv * DC_D + col * 4;
    const T* pa = a_in + row * a_stride + h * DC_D + col * 4;
    f32x4 a, c, e;
    float sa = 0.0f, sc = 0.0f;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      a[x] = ldf(pk + x);
      c[x] = ldf(pq + x);
      e[x] = expf(-rate * softplus_exact(ldf(pa + x) + dt[x]));
      sa += a[x] * a[x];
      sc += c[x] * c[x];
    }
    const float ra = 1.0f / sqrtf(row_sum16(sa) + 1e-6f);
    const float rc = 1.0f / (sqrtf(row_sum16(sc) + 1e-6f) * sqrtf((float)DC_D));
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      a[x] = t < n ? a[x] * ra : 0.0f;
      c[x] = t < n ? c[x] * rc : 0.0f;
      e[x] = t < n ? e[x] : 1.0f;
    }
    *reinterpret_cast<f32x4*>(&k[t][col * 4]) = a;
    *reinterpret_cast<f32x4*>(&q[t][col * 4]) = c;
    *reinterpret_cast<f32x4*>(&g[t][col * 4]) = e;
    const unsigned long long odd = __ballot(not_finite(a) + not_finite(e) != 0.0f);
    if (odd && bad == DC_C) bad = i * 4 + __builtin_ctzll(odd) / 16;
  }
  float strength = 0.0f;
  if (lane < n && lane < DC_C) strength = sigmoid_exact(ldf(beta_logit + (int64_t)(t0 + lane) * beta_stride + h));
  if (lane < DC_C) beta[lane] = strength;
  if (const unsigned long long odd = __ballot(strength - strength != 0.0f)) bad = min(bad, (int)__builtin_ctzll(odd));
  for (int i = lane; i < DC_C * (DC_C + 1); i += WAVE) (&L[0][0])[i] = (&M[0][0])[i] = 0.0f;
  __syncthreads();

  // four s at a time, 16 lanes each, four d a lane: k_s times the decays up to t, against k_t and q_t
#pragma unroll
  for (int sb = 0; sb < 4; ++sb) {
    const int s = sb * 4 + grp;
    f32x4 w = *reinterpret_cast<const f32x4*>(&k[s][col * 4]);
#pragma unroll
    for (int t = sb * 4; t < DC_C; ++t) {
      const f32x4 e = *reinterpret_cast<const f32x4*>(&g[t][col * 4]);
      const f32x4 a = *reinterpret_cast<const f32x4*>(&k[t][col * 4]);
      const f32x4 c = *reinterpret_cast<const f32x4*>(&q[t][col * 4]);
      float l = 0.0f, m = 0.0f;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        w[x] = t > s ? w[x] * e[x] : w[x];
        l += a[x] * w[x];
        m += c[x] * w[x];
      }
      l = row_sum16(l);
      m = row_sum16(m);
      if (col == 0 && t >= s) {
        M[t][s] = m;
        if (t > s) L[t][s] = l * beta[t];
      }
    }
  }
  __syncthreads();

  // column j of the inverse by forward substitution, a lane each
  if (lane < DC_C) {
    float x[DC_C];
#pragma unroll
    for (int t = 0; t < DC_C; ++t) {
      float sum = t == lane ? 1.0f : 0.0f;
#pragma unroll
      for (int s = 0; s < t; ++s) sum -= L[t][s] * x[s];
      x[t] = sum;
      Ti[t][lane] = sum;
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) r0[DC_M + (i * 4 + grp) * DC_C + col] = M[i * 4 + grp][col];
  __syncthreads();

  // the running products, a lane per d
  {
    const int d = lane;
    float p = 1.0f;
    float kk[DC_C];
#pragma unroll
    for (int t = 0; t < DC_C; ++t) {
      kk[t] = k[t][d];
      p *= g[t][d];
      r0[DC_Q + t * DC_D + d] = p * q[t][d];
      k[t][d] = beta[t] * (p * kk[t]);
    }
    r0[DC_P + d] = p;
    p = 1.0f;
#pragma unroll
    for (int t = DC_C - 1; t >= 0; --t) {
      kk[t] *= p;
      p *= g[t][d];
    }
    for (int t = bad; t < DC_C; ++t) k[t][d] = 0.0f;
#pragma unroll
    for (int t = 0; t < DC_C; t += 4)
      *reinterpret_cast<f32x4*>(r0 + DC_K + d * DC_C + t) = f32x4{kk[t], kk[t + 1], kk[t + 2], kk[t + 3]};
  }
  __syncthreads();

  float ti[4];                             // A operand: row col, columns kk * 4 + grp
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) ti[kk] = Ti[col][kk * 4 + grp];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(ti[kk], k[kk * 4 + grp][m * 16 + col], acc, 0, 0, 0);
    if (bad < DC_C) {
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] = grp * 4 + r < bad ? acc[r] : NAN;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) r0[DC_W + (grp * 4 + r) * DC_D + m * 16 + col] = acc[r];
  }
  for (int v0 = 0; v0 < V; v0 += 16) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f}, x;     // x[kk]: token 4 kk + grp
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int s = kk * 4 + grp;
      const float v = ldf(v_in + (int64_t)(t0 + min(s, n - 1)) * v_stride + h * V + v0 + col);
      x[kk] = s < n && s < bad ? beta[s] * v : 0.0f;
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(ti[kk], x[kk] - x[kk] == 0.0f ? x[kk] : 0.0f, acc, 0, 0, 0);
    }
    if (bad < DC_C || __any(not_finite(x) != 0.0f)) {
      f32x4 y;                               // as rows 4 grp + r: token 4 kk + g is in lane group g's x[kk]
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float a = __shfl(x[0], r * 16 + col), b = __shfl(x[1], r * 16 + col), c = __shfl(x[2], r * 16 + col),
                    d = __shfl(x[3], r * 16 + col);
        y[r] = grp == 0 ? a : grp == 1 ? b : grp == 2 ? c : d;
      }
      const int first = min(bad, first_odd_row(y, col));
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] = grp * 4 + r < first ? acc[r] : NAN;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) r0[DC_U + (int64_t)(grp * 4 + r) * V + v0 + col] = acc[r];
  }
}

struct ChunkRegs {                         // a lane's operands of one chunk
  f32x4 w[4], q[4], k[4], m, p[4], u;
};

// 4 waves of 16 value columns
__global__ void __launch_bounds__(4 * WAVE, 1) delta_scan_kernel(float* __restrict__ o, const float* __restrict__ rec,
                                                                 float* __restrict__ state,
                                                                 const int* __restrict__ slots,
                                                                 const int* __restrict__ cu,
                                                                 const int* __restrict__ seg_start, int H, int V) {
  const int b = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
  const int v = (blockIdx.z * 4 + (threadIdx.x >> 6)) * 16 + col;
  if (v - col >= V) return;                // a whole wave: V is a multiple of 16
  const int t0 = cu[b], t1 = cu[b + 1], chunks = (t1 - t0 + DC_C - 1) / DC_C;
  const int64_t size = DC_U + DC_C * V;
  const float* r0 = rec + ((int64_t)chunk_base(cu, b) * H + h) * size;
  float* sp = state + ((int64_t)slots[b] * H + h) * DC_D * V + v;
  f32x4 S[4];                              // d = 16 m + 4 grp + r of column v
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[m][r] = seg_start[b] == 0 ? 0.0f : sp[(int64_t)(m * 16 + grp * 4 + r) * V];
  auto fetch = [&](int c) {
    const float* p = r0 + (int64_t)c * H * size;
    ChunkRegs x;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      x.w[m] = *reinterpret_cast<const f32x4*>(p + DC_W + col * DC_D + m * 16 + grp * 4);
      x.q[m] = *reinterpret_cast<const f32x4*>(p + DC_Q + col * DC_D + m * 16 + grp * 4);
      x.k[m] = *reinterpret_cast<const f32x4*>(p + DC_K + (m * 16 + col) * DC_C + grp * 4);
      x.p[m] = *reinterpret_cast<const f32x4*>(p + DC_P + m * 16 + grp * 4);
      x.u[m] = p[DC_U + (int64_t)(grp * 4 + m) * V + v];
    }
    x.m = *reinterpret_cast<const f32x4*>(p + DC_M + col * DC_C + grp * 4);
    return x;
  };
  auto step = [&](const ChunkRegs& x, int c) {
    f32x4 ws[2] = {}, qs[2] = {};
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        ws[r & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w[m][r], S[m][r], ws[r & 1], 0, 0, 0);
        qs[r & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.q[m][r], S[m][r], qs[r & 1], 0, 0, 0);
      }
    f32x4 u, out;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      u[r] = x.u[r] - (ws[0][r] + ws[1][r]);
      out[r] = qs[0][r] + qs[1][r];
    }
    f32x4 um;                              // what M takes: in time beside the state's chain, which takes u
#pragma unroll
    for (int r = 0; r < 4; ++r) um[r] = u[r] - u[r] == 0.0f ? u[r] : 0.0f;
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[m][r] *= x.p[m][r];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {       // s = 4 grp + kk
      out = __builtin_amdgcn_mfma_f32_16x16x4f32(x.m[kk], um[kk], out, 0, 0, 0);
#pragma unroll
      for (int m = 0; m < 4; ++m) S[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[m][kk], u[kk], S[m], 0, 0, 0);
    }
    if (__any(not_finite(u) != 0.0f)) {
      const int first = first_odd_row(u, col);
#pragma unroll
      for (int r = 0; r < 4; ++r) out[r] = grp * 4 + r < first ? out[r] : NAN;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = t0 + c * DC_C + grp * 4 + r;
      if (t < t1) o[((int64_t)t * H + h) * V + v] = out[r];
    }
  };
  // three chunks of operands: two are on their way while one is multiplied
  ChunkRegs x[3] = {};
#pragma unroll
  for (int i = 0; i < 3; ++i)
    if (i < chunks) x[i] = fetch(i);
#pragma unroll 1
  for (int c = 0; c < chunks; c += 3) {
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (c + i < chunks) {
        step(x[i], c + i);
        if (c + i + 3 < chunks) x[i] = fetch(c + i + 3);
      }
  }
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) sp[(int64_t)(m * 16 + grp * 4 + r) * V] = S[m][r];
}

// floats of rec, or 0 where the token-by-token form is taken: other sizes, steps whose records would take more than 1 GB, and
// short segments, where it ends sooner: below 64 tokens on average (8 x 32 tokens, 16 heads of 64 x 128, 25 us and 35 here; 8 x
// 100 66 and 54), 96 of wide values, whose records are longer (one of 64, 8 heads of 64 x 256, 31 and 37; of 100 45 and 43),
// and 128 where segments and heads fill the chip without chunks (64 segments, 32 heads of 64 x 128: of 64 tokens 307 and
// 331, of 100 483 and 511, of 128 612 and 593)
extern "C" int64_t seq_delta_chunk_room(int T_, int B, int H, int G, int D, int V) {
  const int least = (int64_t)B * H * V >= 1 << 18 ? 128 : V > 128 ? 96 : 64;
  if (D != DC_D || V % 16 != 0 || V < 16 || T_ < least * (int64_t)B || H > 65535) return 0;
  const int64_t n = ((int64_t)T_ / DC_C + B) * H * (DC_U + DC_C * V);
  return n <= (int64_t)1 << 28 ? n : 0;
}

extern "C" void seq_launch_delta_chunks(float* o, const void* q, const void* k, const void* v, const void* beta_logit,
                                        const void* a, const float* dt_bias, const float* a_log, float* rec, float* state,
                                        const int* slots, const int* cu, const int* seg_start, int T_, int B, int H, int G,
                                        int V, int q_stride, int k_stride, int v_stride, int beta_stride, int a_stride,
                                        int is_f32, hipStream_t st) {
#define DC_GO(T)                                                                                                     \
  hipLaunchKernelGGL(delta_chunk_kernel<T>, dim3(T_ / DC_C + B, H), dim3(WAVE), 0, st, rec, (const T*)q, (const T*)k, \
                     (const T*)v, (const T*)beta_logit, (const T*)a, dt_bias, a_log, cu, B, H, G, V, q_stride,       \
                     k_stride, v_stride, beta_stride, a_stride)
  if (is_f32) DC_GO(float);
  else DC_GO(bfraw);
#undef DC_GO
  hipLaunchKernelGGL(delta_scan_kernel, dim3(B, H, (V + 63) / 64), dim3(4 * WAVE), 0, st, o, rec, state, slots, cu, seg_start,
                     H, V);
}
