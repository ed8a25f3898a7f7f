// Paged decode attention (single new token per stream) for gfx950.
//
// Flash decoding over 32-key tiles, one tile per WAVE: a wave takes every
// (Z*4)-th tile of its (stream, kv head), keeps its own running max and sum, and
// the four waves of a workgroup fold once at the end. Z workgroups share a
// context; their partials are merged by a second launch (none with Z = 1).
//
// What bounds it is bytes in flight: a wave issues the K and V loads of a whole
// tile (16 KB in bf16, 64 registers a lane) before it uses any, so twelve waves
// keep 192 KB in flight per compute unit, and no barrier stands between a wave's
// scores, softmax and weighted sum. (64-key tiles leave two waves per SIMD, and
// loading the next tile ahead spills: 43 and 126 us where this takes 36.)
//
//   scores   S[key][head] on the matrix cores (16x16x32): K rows go from memory to
//            fragments as they lie - lane group g takes dims 32g..32g+31 of its
//            row, 64 contiguous bytes in four loads, and Q is read in the same
//            order (a dot product does not care which order its terms have)
//   softmax  fp32, head per lane column, exchanges over the four lane groups only
//   P V      fp32 on the vector unit: 16 lanes x 8 dims span a V row, four keys at
//            a time; P crosses lanes through a wave-private LDS strip
//
// Workgroups are laid out kv head fastest: with 8 kv heads each XCD serves one of
// them, and the streams of a request, neighbours in the batch, find their shared
// prompt's rows in that XCD's L2.
//
// Layouts: q [B, H, D=128]; caches [NB, KVH, BS, D]; block_tables [B, MAXB];
// context_lens INCLUDE the current token. GQA in {1, 2, 4, 8}. Optionally a context sees
// only its last token's aligned block of mask_size positions, and each head's result
// passes a sigmoid gate (the block-local layers of the hybrid family).
//
// Measured with the merge, 32 heads / 8 kv heads, beside 256-key workgroups with
// block-wide passes: 120 streams of 560 keys 36.5 us (68), 5 streams 8.5 us (23), 16
// fp8 streams of 5850 keys 49 us (109, 198 MB: 4 TB/s); 16 / 4 heads, one stream of
// 170 keys 7.8 us (21); block-local, 40 rows of 600 keys, 16 / 4 heads,
// 20.5 us (81 with a workgroup per row and q-head).

#include "common.h"

typedef __bf16 bf16x8_mfma __attribute__((ext_vector_type(8)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

#define NTHREADS 256
#define TKEYS 32           // keys of a wave's tile
// partials layout: [B, KVH, Z, GQA, 130]: 128 o values + m + l
#define PART_STRIDE 130

union Frag {
  u32x4 u;
  bf16x8_mfma m;
};

// 8 fp8 -> 8 bf16 (every e4m3 value is a bf16 value)
__device__ __forceinline__ Frag fp8x8_to_bf16(u32x2 v) {
  Frag f;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)v[i], false);
    const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)v[i], true);
    f.u[2 * i] = __builtin_amdgcn_perm(__float_as_uint(lo[1]), __float_as_uint(lo[0]), 0x07060302u);
    f.u[2 * i + 1] = __builtin_amdgcn_perm(__float_as_uint(hi[1]), __float_as_uint(hi[0]), 0x07060302u);
  }
  return f;
}

// first key that a context of L keys sees: 0, or the start of its last token's aligned
// block of mask_size positions
__device__ __forceinline__ int first_key(int L, int mask_size) {
  return mask_size > 0 ? max(L - 1, 0) / mask_size * mask_size : 0;
}

// LOCAL (block-local layers): exponentials to the last place, as those layers' other kernels
// have them; __expf of an argument of -70 is off by 3e-6. 40 rows of 600 keys, 16 / 4 heads,
// in a graph: 17.0 us, 15.9 with __expf
template <bool LOCAL>
__device__ __forceinline__ float exp_of(float x) {
  return LOCAL ? expf(x) : __expf(x);
}

template <bool LOCAL>
__device__ __forceinline__ float head_gate(const bf16_t* __restrict__ gate, int stride, int b, int h) {
  if (!gate) return 1.0f;
  return 1.0f / (1.0f + exp_of<LOCAL>(-bf16_to_f32(((const short*)gate)[(int64_t)b * stride + h])));
}

template <int GQA, bool FP8, bool LOCAL>
__global__ __launch_bounds__(NTHREADS, GQA == 8 ? 2 : 3) void attn_decode_tiles(
    float* __restrict__ partials, bf16_t* __restrict__ out,  // out: written when gridDim.z == 1
    const bf16_t* __restrict__ q,        // [B, H, 128], row stride q_tstride
    const char* __restrict__ k_cache,    // [NB, KVH, BS, 128], bf16 or fp8
    const char* __restrict__ v_cache,
    const float* __restrict__ k_scale,   // [NB, KVH, BS] per-row dequant (FP8 only)
    const float* __restrict__ v_scale,
    const int* __restrict__ block_tables,  // [B, max_blocks]
    const int* __restrict__ context_lens,  // [B]
    const bf16_t* __restrict__ gate, int gate_stride,  // [B, H] logits of the heads' sigmoid gates, or nullptr
    float scale, int block_size, int max_blocks, int q_tstride, int mask_size) {
  const int g_kv = blockIdx.x, num_kv_heads = gridDim.x;
  const int b = blockIdx.y;
  const int z = blockIdx.z, Z = gridDim.z;
  const int L = context_lens[b];
  const int first = first_key(L, mask_size);
  const int tiles = (L - first + TKEYS - 1) / TKEYS;
  if (z * 4 >= tiles && Z > 1) return;   // no keys here: the merge skips this partial
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int col = lane & 15, grp = lane >> 4;

  __shared__ __attribute__((aligned(16))) float p_lds[4][TKEYS * GQA];
  __shared__ float o_lds[4][GQA * 128];
  __shared__ float m_lds[4][GQA], l_lds[4][GQA];
  float* p_me = p_lds[wave];

  Frag qf[4];
  {
    const short* qp = (const short*)q + (int64_t)b * q_tstride + (g_kv * GQA + min(col, GQA - 1)) * 128 + grp * 32;
#pragma unroll
    for (int s = 0; s < 4; ++s)
      qf[s].u = col < GQA ? *reinterpret_cast<const u32x4*>(qp + s * 8) : u32x4{0, 0, 0, 0};
  }
  const int* bt = block_tables + (int64_t)b * max_blocks;

  float m_run = -INFINITY, l_run = 0.0f;   // of head ``col``; l_run: this lane's keys only
  float o[GQA][8];
#pragma unroll
  for (int h = 0; h < GQA; ++h)
#pragma unroll
    for (int j = 0; j < 8; ++j) o[h][j] = 0.0f;

  // cache row of key first + tile * 32 + (lane & 31); keys behind the context repeat its
  // last row
  auto row_of = [&](int tile) {
    const int kc = min(first + tile * TKEYS + (lane & (TKEYS - 1)), L - 1);
    return (bt[kc / block_size] * num_kv_heads + g_kv) * block_size + kc % block_size;
  };
  const int t0 = z * 4 + wave;
  int row_next = t0 < tiles ? row_of(t0) : 0;
#pragma unroll 1
  for (int t = t0; t < tiles; t += Z * 4) {
    const int base = first + t * TKEYS;
    const int rowi = row_next;
    float ks = 1.0f, vs = 1.0f;
    if constexpr (FP8) { ks = k_scale[rowi]; vs = v_scale[rowi]; }
    u32x4 kraw[TKEYS / 16][FP8 ? 2 : 4];
#pragma unroll
    for (int tt = 0; tt < TKEYS / 16; ++tt) {
      const int64_t r = __shfl(rowi, tt * 16 + col);
      const u32x4* kp = reinterpret_cast<const u32x4*>(k_cache + r * (FP8 ? 128 : 256) + grp * (FP8 ? 32 : 64));
#pragma unroll
      for (int s = 0; s < (FP8 ? 2 : 4); ++s) kraw[tt][s] = kp[s];
    }
    u32x4 vraw[TKEYS / 4];
#pragma unroll
    for (int i = 0; i < TKEYS / 4; ++i) {
      const int64_t r = __shfl(rowi, i * 4 + grp);
      if constexpr (FP8) {
        const u32x2 v = *reinterpret_cast<const u32x2*>(v_cache + r * 128 + col * 8);
        vraw[i][0] = v[0];
        vraw[i][1] = v[1];
      } else {
        vraw[i] = *reinterpret_cast<const u32x4*>(v_cache + r * 256 + col * 16);
      }
    }
    row_next = row_of(min(t + Z * 4, tiles - 1));

    // ---- scores: lane (col, grp) holds keys tt*16 + grp*4 + r of head col ----
    float sc[TKEYS / 16][4];
    float tmax = -INFINITY;
#pragma unroll
    for (int tt = 0; tt < TKEYS / 16; ++tt) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        Frag kf;
        if constexpr (FP8)
          kf = fp8x8_to_bf16(u32x2{kraw[tt][s >> 1][(s & 1) * 2], kraw[tt][s >> 1][(s & 1) * 2 + 1]});
        else
          kf.u = kraw[tt][s];
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf.m, qf[s].m, acc, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = tt * 16 + grp * 4 + r;
        float x = acc[r] * scale;
        if constexpr (FP8) x *= __shfl(ks, key);
        sc[tt][r] = base + key < L ? x : -INFINITY;
        tmax = fmaxf(tmax, sc[tt][r]);
      }
    }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
    const float m_new = fmaxf(m_run, tmax);
    const float alpha = (m_run == -INFINITY) ? 0.0f : exp_of<LOCAL>(m_run - m_new);
    m_run = m_new;
    l_run *= alpha;
#pragma unroll
    for (int tt = 0; tt < TKEYS / 16; ++tt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = (sc[tt][r] == -INFINITY) ? 0.0f : exp_of<LOCAL>(sc[tt][r] - m_new);
        l_run += p;
        if (col < GQA) p_me[(tt * 16 + grp * 4 + r) * GQA + col] = p;
      }
    // the strip is this wave's own: in-order LDS, only the compiler is held
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int h = 0; h < GQA; ++h) {
      const float a = __shfl(alpha, h);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[h][j] *= a;
    }

    // ---- P V: lane (col, grp) adds dims col*8.. of keys i*4 + grp ------------
#pragma unroll
    for (int i = 0; i < TKEYS / 4; ++i) {
      float p[GQA];
#pragma unroll
      for (int h = 0; h < GQA; ++h) p[h] = p_me[(i * 4 + grp) * GQA + h];
      if constexpr (FP8) {
        const float s = __shfl(vs, i * 4 + grp);
#pragma unroll
        for (int h = 0; h < GQA; ++h) p[h] *= s;
      }
      float v[8];
#pragma unroll
      for (int w = 0; w < (FP8 ? 2 : 4); ++w) {
        if constexpr (FP8) {
          const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)vraw[i][w], false);
          const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)vraw[i][w], true);
          v[4 * w] = lo[0];
          v[4 * w + 1] = lo[1];
          v[4 * w + 2] = hi[0];
          v[4 * w + 3] = hi[1];
        } else {
          v[2 * w] = __uint_as_float(vraw[i][w] << 16);
          v[2 * w + 1] = __uint_as_float(vraw[i][w] & 0xffff0000u);
        }
      }
#pragma unroll
      for (int h = 0; h < GQA; ++h)
#pragma unroll
        for (int j = 0; j < 8; ++j) o[h][j] += p[h] * v[j];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }

  // ---- fold the lane groups' keys, then the waves ---------------------------
  l_run += __shfl_xor(l_run, 16);
  l_run += __shfl_xor(l_run, 32);
  // halves, then odd and even rows of 16 lanes: each exchange sums two values and
  // leaves one in either part, so a lane ends with dims 2*grp' and 2*grp'+1 of its
  // eight, grp' = the part it landed in
#pragma unroll
  for (int h = 0; h < GQA; ++h) {
    float half[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(o[h][j]), __float_as_uint(o[h][j + 4]), false, false);
      half[j] = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);   // lanes 0-31: dim j, 32-63: dim j + 4
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(half[j]), __float_as_uint(half[j + 2]), false, false);
      const float v = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);  // even rows: dim j, odd rows: dim j + 2
      o_lds[wave][h * 128 + col * 8 + (lane >> 5) * 4 + (grp & 1) * 2 + j] = v;
    }
  }
  if (lane < GQA) {
    m_lds[wave][lane] = m_run;
    l_lds[wave][lane] = l_run;
  }
  __syncthreads();
  float* base = partials + (((int64_t)b * num_kv_heads + g_kv) * Z + z) * GQA * PART_STRIDE;
  for (int i = tid; i < GQA * 128; i += NTHREADS) {
    const int h = i >> 7, d = i & 127;
    float M = m_lds[0][h];
#pragma unroll
    for (int w = 1; w < 4; ++w) M = fmaxf(M, m_lds[w][h]);
    float acc = 0.0f, l = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float e = m_lds[w][h] == -INFINITY ? 0.0f : exp_of<LOCAL>(m_lds[w][h] - M);   // a wave without a tile
      acc += o_lds[w][i] * e;
      l += l_lds[w][h] * e;
    }
    if (Z == 1) {
      const float v = (l > 0.0f ? acc / l : 0.0f) * head_gate<LOCAL>(gate, gate_stride, b, g_kv * GQA + h);
      ((short*)out)[((int64_t)b * num_kv_heads * GQA + g_kv * GQA + h) * 128 + d] = f32_to_bf16(v);
    } else {
      base[h * PART_STRIDE + d] = acc;
      if (d == 0) {
        base[h * PART_STRIDE + 128] = M;
        base[h * PART_STRIDE + 129] = l;
      }
    }
  }
}

// Workgroups per context: about 640 in all, and never more than the longest
// context has groups of four tiles. Below that the chip is not full, above it the
// merge and the workgroups' fixed part (lengths, table, fold: 4 us) cost more than
// the shorter loops give. With the merge, bf16, 960 (stream, kv head) pairs of 560
// keys: 36.5 us with 1, 42 with 2, 47 with 8; fp8, 128 pairs of 5850 keys: 114 with
// 1, 58 with 3, 49 with 4 to 6, 54 with 24.
extern "C" int attn_decode_splits(int B, int num_kv_heads, int max_ctx) {
  const int most = (max_ctx + 4 * TKEYS - 1) / (4 * TKEYS);
  const int want = (640 + B * num_kv_heads / 2) / (B * num_kv_heads);
  const int z = want < most ? want : most;
  return z < 1 ? 1 : z;
}

// merge the partials of a (stream, q head): two dims per lane, the partials dealt
// to four waves
template <bool LOCAL>
__global__ void __launch_bounds__(256) attn_decode_merge_kernel(
    bf16_t* __restrict__ out,            // [B, H, 128]
    const float* __restrict__ partials,  // [B, KVH, Z, gqa, 130]
    const int* __restrict__ context_lens, const bf16_t* __restrict__ gate, int gate_stride, int gqa, int Z,
    int mask_size) {
  const int b = blockIdx.y, h = blockIdx.x, num_q_heads = gridDim.x;
  const int g_kv = h / gqa, g = h % gqa;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int L = context_lens[b];
  const int tiles = (L - first_key(L, mask_size) + TKEYS - 1) / TKEYS;
  const int n = min(Z, (tiles + 3) / 4);
  const float* base = partials + (((int64_t)b * (num_q_heads / gqa) + g_kv) * Z * gqa + g) * PART_STRIDE;
  const int64_t step = (int64_t)gqa * PART_STRIDE;
  float m = -INFINITY;
  for (int c = lane; c < n; c += 64) m = fmaxf(m, base[c * step + 128]);
  m = wave_reduce_max(m);
  float a0 = 0.0f, a1 = 0.0f, l = 0.0f;
#pragma unroll 4
  for (int c = wave; c < n; c += 4) {
    const float* p = base + c * step;
    const float w = exp_of<LOCAL>(p[128] - m);
    const f32x2 v = *reinterpret_cast<const f32x2*>(p + lane * 2);
    l += p[129] * w;
    a0 += v[0] * w;
    a1 += v[1] * w;
  }
  __shared__ float sh_o[4][128], sh_l[4];
  sh_o[wave][lane * 2] = a0;
  sh_o[wave][lane * 2 + 1] = a1;
  if (lane == 0) sh_l[wave] = l;
  __syncthreads();
  const int d = threadIdx.x;
  if (d < 128) {
    const float acc = sh_o[0][d] + sh_o[1][d] + sh_o[2][d] + sh_o[3][d];
    const float lt = sh_l[0] + sh_l[1] + sh_l[2] + sh_l[3];
    ((short*)out)[((int64_t)b * num_q_heads + h) * 128 + d] = f32_to_bf16((lt > 0.0f ? acc / lt : 0.0f) * head_gate<LOCAL>(gate, gate_stride, b, h));
  }
}

// Rows of one launch: they lie on the grid's y, which ends at 65535. Steps with a row
// per token (prompt portions on the fp8 cache, short segments) can have more and go out
// in several launches; on x, beside the kv heads, every workgroup would divide.
#define MAX_ROWS 65535

// picks the GQA instantiation (the binding admits 1, 2, 4, 8); mask_size: -1 plain decode,
// from 0 on a block-local layer's (bf16 caches); partials: room for
// min(B, MAX_ROWS) * KVH * splits * gqa * 130 floats when splits > 1
extern "C" void launch_attn_decode(
    bf16_t* out, float* partials, const bf16_t* q, const void* k_cache, const void* v_cache,
    const float* k_scale, const float* v_scale, const int* block_tables, const int* context_lens,
    const bf16_t* gate, int gate_stride, float scale, int num_q_heads, int num_kv_heads, int block_size,
    int max_blocks, int splits, int q_tstride, int B, int cache_fp8, int mask_size, hipStream_t stream) {
  const int gqa = num_q_heads / num_kv_heads;
  const bool local = mask_size >= 0;
  for (int b0 = 0; b0 < B; b0 += MAX_ROWS) {
    const int rows = B - b0 < MAX_ROWS ? B - b0 : MAX_ROWS;
    const dim3 grid(num_kv_heads, rows, splits);
    bf16_t* o = out + (int64_t)b0 * num_q_heads * 128;
    const bf16_t* q0 = q + (int64_t)b0 * q_tstride;
    const int* bt = block_tables + (int64_t)b0 * max_blocks;
    const bf16_t* g0 = gate ? gate + (int64_t)b0 * gate_stride : nullptr;
#define LAUNCH(G, F, L)                                                                            \
  hipLaunchKernelGGL((attn_decode_tiles<G, F, L>), grid, dim3(NTHREADS), 0, stream, partials, o, q0, \
                     (const char*)k_cache, (const char*)v_cache, k_scale, v_scale, bt,             \
                     context_lens + b0, g0, gate_stride, scale, block_size, max_blocks, q_tstride, mask_size)
#define DISPATCH(G) \
  do { if (cache_fp8) LAUNCH(G, true, false); else if (local) LAUNCH(G, false, true); else LAUNCH(G, false, false); } while (0)
    switch (gqa) {
      case 1: DISPATCH(1); break;
      case 2: DISPATCH(2); break;
      case 4: DISPATCH(4); break;
      default: DISPATCH(8); break;
    }
#undef DISPATCH
#undef LAUNCH
    if (splits > 1)
      hipLaunchKernelGGL(local && !cache_fp8 ? attn_decode_merge_kernel<true> : attn_decode_merge_kernel<false>,
                         dim3(num_q_heads, rows), dim3(256), 0, stream, o, partials, context_lens + b0, g0,
                         gate_stride, gqa, splits, mask_size);
  }
}
