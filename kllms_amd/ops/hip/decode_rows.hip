// The row-wise steps between the products of a decode step, for gfx950: what a step
// of up to 128 rows does there is launch latency (4.7 us a kernel in a replayed
// graph) and little else, so each of these kernels does all the work that lies
// between two products, and takes the previous product's fp32 split sums as they are
// (linear_rows.hip), which saves the reduction's launch. The sums are rounded to bf16
// where a whole product's result would be: these products of a step of few rows and of
// one of many then agree to the last bits of their sums. (Not so gate and up: with the
// activation in the product they stay in fp32, from the library they come in bf16.)
//
// Per layer: residual + norm (twice) and rope + cache store, beside attention and
// four products: 8 launches (one more where gate/up is the library's), where separate reductions, rope, store and activation
// took 11. A step of 5 rows (32 heads, width 4096, 6 layers, contexts of 560) went
// from 948 to 774 us with these and few-row products through registers, and to 676 with those of linear_rows.hip; one of
// 120 rows from 1516 to 1237 and 1114, one of a single row at width 2048 from 492 to 391 and 330. (With the merge in
// attention's launch and weights that pass the caches by they are at 612, 1024 and 284.)

#include <type_traits>

#include "common.h"

#define DR_THREADS 1024

// Sum of the splits of part [S, ...] at `at`, in their order. The loads of two, four or eight splits go out together, those
// past the last one to its place: a loop over S waits for each load by itself where S is no multiple of what is unrolled (the
// steps above with such a loop: 688, and 344 for the single row).
template <int B, typename V>
__device__ __forceinline__ V splits_of(const float* __restrict__ part, int s0, int S, int64_t plane, int64_t at, V sum) {
  V v[B];
#pragma unroll
  for (int s = 0; s < B; ++s) v[s] = *reinterpret_cast<const V*>(part + min(s0 + s, S - 1) * plane + at);
#pragma unroll
  for (int s = 0; s < B; ++s)
    if (s0 + s < S) sum += v[s];
  return sum;
}
template <typename V>
__device__ __forceinline__ V split_sum(const float* __restrict__ part, int S, int64_t plane, int64_t at) {
  const V zero = {};
  if (S <= 2) return splits_of<2>(part, 0, S, plane, at, zero);
  if (S <= 4) return splits_of<4>(part, 0, S, plane, at, zero);
  V sum = splits_of<8>(part, 0, S, plane, at, zero);
  for (int s0 = 8; s0 < S; s0 += 8) sum = splits_of<8>(part, s0, S, plane, at, sum);
  return sum;
}

// Sum over the workgroup, for all its threads. The chain of a row runs through it: register moves within a wave and one
// barrier, where shuffles through LDS and two took 0.6 us longer.
__device__ __forceinline__ float row_sum(float v, float* scratch) {
  auto moved = [](float x, auto how) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), decltype(how)::value, 0xf, 0xf, false));
  };
  auto over_wave = [&](float x, bool halves) {
    x += moved(x, std::integral_constant<int, 0xb1>());    // quad_perm 1 0 3 2
    x += moved(x, std::integral_constant<int, 0x4e>());    // quad_perm 2 3 0 1
    x += moved(x, std::integral_constant<int, 0x141>());   // row_half_mirror
    x += moved(x, std::integral_constant<int, 0x140>());   // row_mirror
    if (!halves) return x;
    const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(s[0]) + __uint_as_float(s[1]);
    const auto t = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(t[0]) + __uint_as_float(t[1]);
  };
  v = over_wave(v, true);
  if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
  __syncthreads();
  return over_wave(scratch[threadIdx.x & 15], false);      // 16 waves
}

// residual[m] += sum of splits (written back, bf16), or residual[m] = table[ids[m]]
// (EMBED, which also zeroes ``clear``); out[m] = rms(residual[m]) * w. One workgroup per row, the row in registers:
// rows of up to 4 * DR_THREADS * VECS elements.
template <bool EMBED, int VECS>
__global__ void __launch_bounds__(DR_THREADS) add_norm_rows_kernel(
    bf16_t* __restrict__ out, bf16_t* __restrict__ residual, const float* __restrict__ part,
    const int64_t* __restrict__ ids, const bf16_t* __restrict__ table, const bf16_t* __restrict__ w, int S, int M,
    int n, int64_t vocab, float eps, int* __restrict__ unknown, int* __restrict__ clear, int clears) {
  __shared__ float red[16];
  if constexpr (EMBED)
    for (int i = blockIdx.x * DR_THREADS + threadIdx.x; i < clears; i += gridDim.x * DR_THREADS) clear[i] = 0;
  const int m = blockIdx.x, tid = threadIdx.x;
  const int nvec = n / 4;
  bf16x4_vec* rv = reinterpret_cast<bf16x4_vec*>(residual + (int64_t)m * n);
  bf16x4_vec* ov = reinterpret_cast<bf16x4_vec*>(out + (int64_t)m * n);
  const bf16x4_vec* wv = reinterpret_cast<const bf16x4_vec*>(w);
  const int64_t id = EMBED ? ids[m] : 0;
  // an id without a row: NaN, never another's memory, and *unknown set for the host
  const bool known = id >= 0 && id < vocab;
  if (EMBED && !known && unknown && tid == 0) __hip_atomic_store(unknown, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  f32x4 x[VECS];
  bf16x4_vec g[VECS];
  float ss = 0.0f;
#pragma unroll
  for (int k = 0; k < VECS; ++k) {
    const int i = tid + k * DR_THREADS;
    if (i >= nvec) break;
    g[k] = wv[i];
    bf16x4_vec r;
    if constexpr (EMBED) {
      r = known ? reinterpret_cast<const bf16x4_vec*>(table + id * n)[i] : bf16x4_vec{0x7fc0, 0x7fc0, 0x7fc0, 0x7fc0};
    } else {
      r = rv[i];
      const f32x4 a = split_sum<f32x4>(part, S, (int64_t)M * n, (int64_t)m * n + i * 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) r[j] = f32_to_bf16(bf16_to_f32(r[j]) + bf16_to_f32(f32_to_bf16(a[j])));
    }
    rv[i] = r;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      x[k][j] = bf16_to_f32(r[j]);
      ss += x[k][j] * x[k][j];
    }
  }
  ss = row_sum(ss, red);
  const float inv = rsqrtf(ss / n + eps);
#pragma unroll
  for (int k = 0; k < VECS; ++k) {
    const int i = tid + k * DR_THREADS;
    if (i >= nvec) break;
    bf16x4_vec o;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = f32_to_bf16(x[k][j] * inv * bf16_to_f32(g[k][j]));
    ov[i] = o;
  }
}

extern "C" void launch_add_norm_rows(bf16_t* out, bf16_t* residual, const float* part, const int64_t* ids,
                                     const bf16_t* table, const bf16_t* w, int S, int M, int n, int64_t vocab,
                                     float eps, int* unknown, int* clear, int clears, hipStream_t stream) {
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(M), dim3(DR_THREADS), 0, stream, out, residual, part, ids, table, w, S, M, n, vocab, eps,
                       unknown, clear, clears);
  };
  const bool narrow = n <= 4 * DR_THREADS;
  if (ids) narrow ? go(add_norm_rows_kernel<true, 1>) : go(add_norm_rows_kernel<true, 4>);
  else narrow ? go(add_norm_rows_kernel<false, 1>) : go(add_norm_rows_kernel<false, 4>);
}

// qkv sums [S, M, (H + 2G) * 128] (+ bias): q and k rotated (entry i with i + 64), q
// out as bf16 rows, k and v into the paged cache - as bf16, or as e4m3 with a scale
// per row (amax / 448 of the bf16 row). A wave per (row, head), two dims a lane.
template <bool FP8>
__global__ void __launch_bounds__(256) rope_store_rows_kernel(
    bf16_t* __restrict__ q_out, const float* __restrict__ part, const bf16_t* __restrict__ bias,
    const int64_t* __restrict__ positions, const float* __restrict__ cos_sin, void* __restrict__ k_cache,
    void* __restrict__ v_cache, float* __restrict__ k_scale, float* __restrict__ v_scale,
    const int64_t* __restrict__ slots, int S, int M, int H, int G, int block_size) {
  const int m = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int head = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (head >= H + 2 * G) return;
  const int N = (H + 2 * G) * 128;
  const int64_t MN = (int64_t)M * N;
  // what is not the sums' is asked for before them
  const bool turned = head < H + G;
  const int64_t slot = head < H ? 0 : slots[m];
  float c = 0.0f, sn = 0.0f, lo_bias = 0.0f, hi_bias = 0.0f;
  if (turned) {
    const float* cs = cos_sin + positions[m] * 128;
    c = cs[lane];
    sn = cs[64 + lane];
  }
  if (bias) {
    lo_bias = bf16_to_f32(((const short*)bias)[head * 128 + lane]);
    hi_bias = bf16_to_f32(((const short*)bias)[head * 128 + lane + 64]);
  }
  const int64_t at = (int64_t)m * N + head * 128 + lane;
  float a = split_sum<float>(part, S, MN, at), b = split_sum<float>(part + 64, S, MN, at);
  if (bias) {
    a += lo_bias;
    b += hi_bias;
  }
  a = bf16_to_f32(f32_to_bf16(a));
  b = bf16_to_f32(f32_to_bf16(b));
  if (turned) {
    const float x = a, y = b;
    a = x * c - y * sn;
    b = y * c + x * sn;
  }
  const short lo = f32_to_bf16(a), hi = f32_to_bf16(b);
  if (head < H) {
    short* o = (short*)q_out + ((int64_t)m * H + head) * 128;
    o[lane] = lo;
    o[lane + 64] = hi;
    return;
  }
  const bool is_k = head < H + G;
  const int g = head - H - (is_k ? 0 : G);
  const int64_t row = ((slot / block_size) * G + g) * block_size + slot % block_size;
  if constexpr (FP8) {
    const float x = bf16_to_f32(lo), y = bf16_to_f32(hi);
    const float sc = fmaxf(wave_reduce_max(fmaxf(fabsf(x), fabsf(y))) * (1.0f / 448.0f), 1e-8f);
    const float inv = 1.0f / sc;
    unsigned char* o = (unsigned char*)(is_k ? k_cache : v_cache) + row * 128;
    o[lane] = f32_to_fp8(x * inv);
    o[lane + 64] = f32_to_fp8(y * inv);
    if (lane == 0) (is_k ? k_scale : v_scale)[row] = sc;
  } else {
    short* o = (short*)(is_k ? k_cache : v_cache) + row * 128;
    o[lane] = lo;
    o[lane + 64] = hi;
  }
}

extern "C" void launch_rope_store_rows(bf16_t* q_out, const float* part, const bf16_t* bias, const int64_t* positions,
                                       const float* cos_sin, void* k_cache, void* v_cache, float* k_scale,
                                       float* v_scale, const int64_t* slots, int S, int M, int H, int G,
                                       int block_size, int fp8, hipStream_t stream) {
  const dim3 grid((H + 2 * G + 3) / 4, M);
  if (fp8)
    hipLaunchKernelGGL(rope_store_rows_kernel<true>, grid, dim3(256), 0, stream, q_out, part, bias, positions,
                       cos_sin, k_cache, v_cache, k_scale, v_scale, slots, S, M, H, G, block_size);
  else
    hipLaunchKernelGGL(rope_store_rows_kernel<false>, grid, dim3(256), 0, stream, q_out, part, bias, positions,
                       cos_sin, k_cache, v_cache, k_scale, v_scale, slots, S, M, H, G, block_size);
}

// Inputs of a captured decode step, in one launch (twelve copies and fills otherwise):
// rows [0, B) from the caller's tensors, [B, bs) padding on the scratch block, block
// tables widened from nb to mb columns with it.
__global__ void __launch_bounds__(256) decode_inputs_kernel(
    int64_t* __restrict__ ids, int64_t* __restrict__ positions, int64_t* __restrict__ slots, int* __restrict__ ctx,
    int* __restrict__ tables, const int64_t* __restrict__ ids_in, const int64_t* __restrict__ positions_in,
    const int64_t* __restrict__ slots_in, const int* __restrict__ ctx_in, const int* __restrict__ tables_in,
    int B, int nb, int mb, int scratch_block, int block_size) {
  const int b = blockIdx.x;
  const bool real = b < B;
  for (int i = threadIdx.x; i < mb; i += 256)
    tables[(int64_t)b * mb + i] = real && i < nb ? tables_in[(int64_t)b * nb + i] : scratch_block;
  if (threadIdx.x == 0) {
    ids[b] = real ? ids_in[b] : 0;
    positions[b] = real ? positions_in[b] : 0;
    slots[b] = real ? slots_in[b] : (int64_t)scratch_block * block_size;
    ctx[b] = real ? ctx_in[b] : 1;
  }
}

extern "C" void launch_decode_inputs(int64_t* ids, int64_t* positions, int64_t* slots, int* ctx, int* tables,
                                     const int64_t* ids_in, const int64_t* positions_in, const int64_t* slots_in,
                                     const int* ctx_in, const int* tables_in, int B, int bs, int nb, int mb,
                                     int scratch_block, int block_size, hipStream_t stream) {
  hipLaunchKernelGGL(decode_inputs_kernel, dim3(bs), dim3(256), 0, stream, ids, positions, slots, ctx, tables, ids_in,
                     positions_in, slots_in, ctx_in, tables_in, B, nb, mb, scratch_block, block_size);
}
