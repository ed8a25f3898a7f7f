// Paged decode attention (single new token per stream) for gfx950.
//
// Flash decoding over 32-key tiles, one tile per WAVE: a wave takes every
// (Z*4)-th tile of its (stream, kv head), keeps its own running max and sum, and
// the four waves of a workgroup fold once at the end. Z workgroups share a
// context (attn_decode_shares); their partials are merged by the last of them to
// arrive, or by a second launch where the caller has no counters for that.
//
// What bounds it is bytes in flight, and for contexts that lie in the L2 the address
// units. A wave has the K and V rows of its next tile (16 KB in bf16, 64 registers a
// lane) on their way while it works on one, twelve waves a compute unit. Rows are read
// whole, 16 neighbouring lanes each (with the fragments' own pattern, four lanes in
// four rows, an instruction occupies the address unit for 64 cycles and not 16), and
// turned by way of a strip of LDS that is the wave's own: no barriers.
//
//   scores   S[key][column] on the matrix cores (16x16x32); column n is head n % GQA
//   softmax  fp32, head per lane column, exchanges over the four lane groups only
//   P V      on the matrix cores: P in three bf16 parts, which are its 32 bits, in
//            columns of their own: n / GQA is the part. The scores' lanes hold P as
//            the product reads it; V comes turned from the strip (ds_read_b64_tr_b16).
//            On the vector unit P V was 360 of a tile's 550 instructions
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
// Measured in graphs, 32 heads / 8 kv heads, against rows read as fragments, P V on the vector unit and merges in a launch of
// their own, us, without the streaming hint (DECODE_ONCE): 120 streams, five to a prompt, of 560 keys 33.5, 25.1; 40, eight to
// a prompt, of 2000 41, 28; prompts of their own: 128 streams of 700 77, 71 (5.5 TB/s), 24 of 2500 48.6, 42.4; 16 fp8 streams of
// 6000 45.5, 40; 5 streams of 560 8.4, 7.4; 16 / 4 heads, one of 150 7.5, 5.6; block-local, 100 rows of 600, 16 / 4 heads 15.5,
// 11.5.
//
// Without groups of heads P V is a quarter of the vector work, and stays on the vector unit: a lane loads the V rows of the keys
// whose scores it has, P is where it is needed, and V needs no strip. 8 / 8 heads, us with the fragments' own loads, by way of the
// matrix cores and so: one stream of 2000 8.0, 8.8, 7.2; 16 of 2000 31.9, 25.3, 24.8; 40 of 500 22.1, 19.9, 18.2; fp8: one of 2000
// 7.2, 8.4, 7.0; 40 of 500 14.0, 14.1, 12.6; 120 of 20, which is four waves to a SIMD or three 5.4, 8.0, 5.4.
//
// Where two heads have a kv head the vector unit's form needs 160 registers, three waves to a SIMD as well, and is 1 % faster in
// bf16 and 3 % slower in fp8 (290 sizes). Against the fragments' own loads, us over sizes drawn up to 3000 keys and 260 streams: 311
// without groups 11 % less, 289 of two heads 11 %, 226 of four 17 %, 74 of eight 27 %. Slower by more than 3 % are a tenth of those
// without groups, by 6 % on average, and an eighth of those of two heads, by 12 %: most of them fp8 caches, or contexts of less than
// 128 keys with more than the 768 workgroups that are there at once. 64 / 32 heads, 57 of 17 9.1, 10.6; fp8, 97 of 41 16.7, 19.5.

#include <algorithm>
#include <type_traits>

#include "common.h"

typedef __bf16 bf16x8_mfma __attribute__((ext_vector_type(8)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4_cvt __attribute__((ext_vector_type(4)));

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
    f.u[2 * i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)v[i], 1.0f, false));
    f.u[2 * i + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)v[i], 1.0f, true));
  }
  return f;
}

// first key that a context of L keys sees: 0, or the start of its last token's aligned
// block of mask_size positions
__device__ __forceinline__ int first_key(int L, int mask_size) {
  return mask_size > 0 ? max(L - 1, 0) / mask_size * mask_size : 0;
}

// How many workgroups share a context of so many rounds of four tiles, a tile for each wave (attn_decode_shares): one up to
// ``few`` rounds. Above, the last of ``most`` from whose ``from`` on it is, no more than ``lo`` or one for every ``per`` rounds,
// and of those as many as are all equally long. ``near``: the least of ``most`` for a context whose prompt a neighbour shares.
struct DecodeShares {
  int few, lo, per, most[3], from[3], near;
  int grid;                  // of no context more
  bool joined;               // merged in the same launch
};
__host__ __device__ __forceinline__ int most_of(int rounds, const DecodeShares& s, bool shared) {
  int z = (rounds + s.per - 1) / s.per, most = rounds >= s.from[1] ? s.most[1] : s.most[0];
  most = rounds >= s.from[2] ? s.most[2] : most;
  z = z < s.lo ? s.lo : z;
  z = z < most ? z : most;
  return shared && z < s.near ? s.near : z;
}
__host__ __device__ __forceinline__ int shares_of(int tiles, const DecodeShares& s, bool shared) {
  const int rounds = (tiles + 3) / 4;
  if (rounds <= s.few) return 1;
  const int z = most_of(rounds, s, shared), each = (rounds + z - 1) / z;
  return (rounds + each - 1) / each;
}

// LOCAL (block-local layers): exponentials to the last place, as those layers' other kernels
// have them; __expf of an argument of -70 is off by 3e-6. 40 rows of 600 keys, 16 / 4 heads,
// in a graph: 17.0 us, 15.9 with __expf
template <bool LOCAL>
__device__ __forceinline__ float exp_of(float x) {
  return LOCAL ? expf(x) : __expf(x);
}

// v of lane from + more
__device__ __forceinline__ int lane_value(int v, int from, int more) { return __builtin_amdgcn_ds_bpermute(from * 4 + more * 4, v); }

template <bool LOCAL>
__device__ __forceinline__ float head_gate(const bf16_t* __restrict__ gate, int stride, int b, int h) {
  if (!gate) return 1.0f;
  return 1.0f / (1.0f + exp_of<LOCAL>(-bf16_to_f32(((const short*)gate)[(int64_t)b * stride + h])));
}

#define MERGED 16          // partials of a thread that are on their way at once when they are merged in the same launch
#define FAR 16             // loads and stores past the L2, from and to other XCDs' workgroups

// A wave's strip of LDS: K of its tile, then V, 32 rows of 128 bf16; after the last one its sums, rows of SUM_PITCH floats
#define SUM_PITCH 132
template <int GQA>
struct Strip {
  static constexpr int SETS = GQA == 8 ? 2 : 1;               // sets of 16 columns
  static constexpr int SUMS = 3 * GQA * SUM_PITCH * 4;
  static constexpr int BYTES = ((SUMS > TKEYS * 256 ? SUMS : TKEYS * 256) + 255) / 256 * 256;
};

// Bytes of a layer's keys and values from which on they are loaded with the streaming hint (nt), unless the stream before or
// behind this one begins with the same block: a shared prompt is read again, from the L2. Layers of as much do not lie in the
// last-level cache (256 MB) any more when the next step comes to them. Steps of six layers, 32 / 8 heads, us without and with:
// 128 streams of 700 1297, 1225; 24 of 2500 910, 881; 40 of 600 794, 782; 8 of 1500 655, 652; one of 7800 629, 617; 16 fp8 streams of
// 6000 857, 830. Prompts of 3000 shared by eight streams each with the hint 941, without 892.
#define DECODE_ONCE (16 << 20)

// KV: what the cache holds
enum { KV_BF16 = 0, KV_FP8 = 1, KV_FP8_ANY = 2 };   // fp8 in blocks of a multiple of four keys, and in others

template <int GQA, int KV, bool LOCAL, bool ONCE>
__device__ __forceinline__ void decode_share(
    float* __restrict__ partials,
    bf16_t* __restrict__ out,            // written where one workgroup has the context, or by the last one with ``arrived``
    const bf16_t* __restrict__ q,        // [B, H, 128], row stride q_tstride
    const char* __restrict__ k_cache,    // [NB, KVH, BS, 128], bf16 or fp8
    const char* __restrict__ v_cache,
    const float* __restrict__ k_scale,   // [NB, KVH, BS] per-row dequant (FP8 only)
    const float* __restrict__ v_scale,
    const int* __restrict__ block_tables,  // [B, max_blocks]
    const int* __restrict__ context_lens,  // [B]
    const bf16_t* __restrict__ gate, int gate_stride,  // [B, H] logits of the heads' sigmoid gates, or nullptr
    int* __restrict__ arrived, int apart,  // [B, KVH] zeros, ``apart`` ints from each other, zeros again afterwards, or nullptr
    float scale, int block_size, uint32_t block_inverse, int max_blocks, int q_tstride, int mask_size, DecodeShares shares,
    int L, int first, int tiles, int Z, char (&strips)[4][Strip<GQA>::BYTES], float (&m_lds)[4][GQA], float (&l_lds)[4][GQA]) {
  constexpr int SETS = Strip<GQA>::SETS;
  constexpr bool FP8 = KV != KV_BF16, ONE = GQA == 1;
  const int g_kv = blockIdx.x, num_kv_heads = gridDim.x;
  const int b = blockIdx.y;
  const int z = blockIdx.z;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // asked for anew behind the loop, whose registers are all taken
  auto lane_now = [] {
    int all = -1;
    asm volatile("" : "+s"(all));
    return (int)__builtin_amdgcn_mbcnt_hi(all, __builtin_amdgcn_mbcnt_lo(all, 0));
  };
  const int lane = lane_now(), col = lane & 15, grp = lane >> 4;

  char* const strip = strips[wave];

  // column n of the products is head n % GQA
  Frag qf[4];
  {
    const short* qp = (const short*)q + (int64_t)b * q_tstride + (g_kv * GQA + col % GQA) * 128 + grp * 8;
#pragma unroll
    for (int s = 0; s < 4; ++s) qf[s].u = *reinterpret_cast<const u32x4*>(qp + s * 32);
  }
  const int* bt = block_tables + (int64_t)b * max_blocks;

  float m_run = -INFINITY, l_run = 0.0f;   // of head col % GQA; l_run: this lane's keys only
  f32x4 o[SETS][8];                      // ONE: the first DIMS floats are this lane's dims, of its keys alone
  constexpr int DIMS = FP8 ? 16 : 8;
#pragma unroll
  for (int e = 0; e < SETS; ++e)
#pragma unroll
    for (int i = 0; i < 8; ++i) o[e][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  // key first + tile * 32 + (lane & 31); those behind the context repeat its last one
  auto key_of = [&](int tile) { return min(first + tile * TKEYS + (lane & (TKEYS - 1)), L - 1); };
  // key / block_size by its reciprocal, which is off by one at most
  auto block_of = [&](int key) {
    const int n = (int)__umulhi((uint32_t)key, block_inverse), rest = key - n * block_size;
    return n - (rest < 0) + (rest >= block_size);
  };
  auto row_of = [&](int tile, int block) {
    const int key = key_of(tile);
    return (block * num_kv_heads + g_kv) * block_size + (key - block_of(key) * block_size);
  };
  typedef __attribute__((address_space(3))) char* lds_t;
  typedef __attribute__((address_space(3))) u32x4* lds_vec;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_t)strip;
  const int row8 = FP8 ? lane >> 3 : grp, turn_row = grp * 4 + (col >> 2);
  // where this lane's 16 bytes of the strip lie: stored, read as K (row col), read turned as V. The rest is an XOR
  uint32_t put_at = lds0 + row8 * 256 + (((FP8 ? (lane & 7) * 2 : col) ^ row8) << 4);
  uint32_t key_at = lds0 + col * 256 + ((grp ^ col) << 4);
  uint32_t turn_at = lds0 + turn_row * 256 + ((((col & 3) >> 1) ^ turn_row) << 4) + (col & 1) * 8;
  // Whole rows go to registers, 16 lanes each (8 in fp8), and from there to the strip, their 16-byte units XORed with the row
  // (ONE: V's stay there, a lane's are of the keys whose scores it has)
  constexpr int LOADS = FP8 ? TKEYS / 8 : TKEYS / 4;
  u32x4 kraw[LOADS], vraw[LOADS];
  f32x4 ks[2], vs[2];                    // scales of this lane's keys tt*16 + grp*4 + r
  auto load = [&](u32x4 (&to)[LOADS], const char* cache, int row, auto own) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      int64_t r;
      if constexpr (!own) r = lane_value(row, FP8 ? lane >> 3 : grp, i * (FP8 ? 8 : 4));
      else if constexpr (FP8) r = lane_value(row, grp * 4 + (lane >> 3 & 1), (i >> 1) * 16 + (i & 1) * 2);
      else r = lane_value(row, grp * 4, (i >> 2) * 16 + (i & 3));
      const u32x4* at = reinterpret_cast<const u32x4*>(cache + (FP8 ? r * 128 + (lane & 7) * 16 : r * 256 + col * 16));
      if constexpr (ONCE) to[i] = __builtin_nontemporal_load(at);
      else to[i] = *at;
    }
  };
  auto load_scales = [&](f32x4 (&to)[2], const float* scales, int row) {
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      if constexpr (KV == KV_FP8) {        // whole quads: of the last one also what lies behind the context
        to[tt] = *reinterpret_cast<const f32x4*>(scales + (lane_value(row, grp * 4, tt * 16) & ~3));
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) to[tt][r] = scales[lane_value(row, grp * 4, tt * 16 + r)];
      }
    }
  };
  auto load_k = [&](int row, auto scales) {
    if constexpr (FP8 && scales) load_scales(ks, k_scale, row);
    load(kraw, k_cache, row, std::false_type());
  };
  auto load_v = [&](int row) {
    if constexpr (FP8) load_scales(vs, v_scale, row);
    load(vraw, v_cache, row, std::bool_constant<ONE>());
  };
  auto store = [&](const u32x4 (&from)[LOADS]) {
    const uint32_t put = put_at;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      if constexpr (FP8) {
        const uint32_t at = put ^ ((i & 1) << 7);
        *(lds_vec)(uintptr_t)(at + i * 2048) = fp8x8_to_bf16(u32x2{from[i][0], from[i][1]}).u;
        *(lds_vec)(uintptr_t)((at ^ 16) + i * 2048) = fp8x8_to_bf16(u32x2{from[i][2], from[i][3]}).u;
      } else {
        *(lds_vec)(uintptr_t)((put ^ ((i & 3) << 6)) + i * 1024) = from[i];
      }
    }
  };
  // the strip is this wave's own: in-order LDS, only the compiler is held
  auto hold = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  const int step = Z * 4;
  int t = z * 4 + wave, row = 0, block = 0;  // row of this lane's key in the next tile; the block of the one behind it
  auto tile = [&](auto more) {
    const int base = first + t * TKEYS;
    // not eighteen addresses for the whole loop
    asm volatile("" : "+v"(put_at), "+v"(key_at), "+v"(turn_at));
    // ---- scores: lane (col, grp) holds keys tt*16 + grp*4 + r of head col % GQA ----
    store(kraw);
    // ONE: the scales themselves, which are loaded anew behind their use: registers for a fourth wave
    const f32x4 ks_now[2] = {ks[0], ks[1]}, vs_now[2] = {vs[0], vs[1]};
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (more) {
      row = row_of(t + step, block);
      block = bt[block_of(key_of(min(t + 2 * step, tiles - 1)))];
      load_k(row, std::bool_constant<!ONE>());
    }
    hold();
    __builtin_amdgcn_sched_barrier(0);
    float sc[TKEYS / 16][4];
    float tmax = -INFINITY;
#pragma unroll
    for (int tt = 0; tt < TKEYS / 16; ++tt) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        Frag kf;
        kf.u = *(lds_vec)(uintptr_t)((key_at ^ (s << 6)) + tt * 4096);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf.m, qf[s].m, acc, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float x = acc[r] * scale;
        if constexpr (FP8) x *= ONE ? ks[tt][r] : ks_now[tt][r];
        sc[tt][r] = base + tt * 16 + grp * 4 + r < L ? x : -INFINITY;
        tmax = fmaxf(tmax, sc[tt][r]);
      }
    }
    if constexpr (more && FP8 && ONE) load_scales(ks, k_scale, row);
    if constexpr (!ONE) {
      hold();
      __builtin_amdgcn_sched_barrier(0);
      store(vraw);
      if constexpr (more) load_v(row);
      __builtin_amdgcn_sched_barrier(0);
    }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
    const float m_new = fmaxf(m_run, tmax);
    if (__any(m_new > m_run)) {
      const float alpha = (m_run == -INFINITY) ? 0.0f : exp_of<LOCAL>(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int e = 0; e < SETS; ++e)
#pragma unroll
        for (int i = 0; i < (ONE ? DIMS / 4 : 8); ++i) o[e][i] *= alpha;
    }
    m_run = m_new;
    if constexpr (ONE) {
#pragma unroll
      for (int tt = 0; tt < TKEYS / 16; ++tt) {
        float p[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          p[r] = (sc[tt][r] == -INFINITY) ? 0.0f : exp_of<LOCAL>(sc[tt][r] - m_new);
          l_run += p[r];
          if constexpr (FP8) p[r] = base + tt * 16 + grp * 4 + r < L ? p[r] * vs[tt][r] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < LOADS / 2; ++i) {
          const u32x4 v = vraw[tt * (LOADS / 2) + i];
          const float even = p[FP8 ? i * 2 : i], odd = p[FP8 ? i * 2 + 1 : i], w = FP8 && lane & 8 ? odd : even;
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            if constexpr (FP8) {
              const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)v[u], false), hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)v[u], true);
              o[0][u] += w * f32x4{lo[0], lo[1], hi[0], hi[1]};
            } else {
              o[0][u >> 1][(u & 1) * 2] += w * __uint_as_float(v[u] << 16);
              o[0][u >> 1][(u & 1) * 2 + 1] += w * __uint_as_float(v[u] & 0xffff0000u);
            }
          }
        }
      }
      if constexpr (more) load_v(row);
      hold();
      __builtin_amdgcn_sched_barrier(0);
      return;
    }
    // P in three bf16 parts, which are its 32 bits: column n of the product has part n / GQA
    Frag pf[SETS];
#pragma unroll
    for (int tt = 0; tt < TKEYS / 16; ++tt) {
      float part[3][4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float p = (sc[tt][r] == -INFINITY) ? 0.0f : exp_of<LOCAL>(sc[tt][r] - m_new);
        l_run += p;
        // scales behind the context are what another sequence left there, infinities too
        if constexpr (FP8) p = base + tt * 16 + grp * 4 + r < L ? p * vs_now[tt][r] : 0.0f;
        part[0][r] = p;
      }
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const f32x4 x = {part[e][0], part[e][1], part[e][2], part[e][3]};
        const u32x2 packed = __builtin_bit_cast(u32x2, __builtin_convertvector(x, bf16x4_cvt));
#pragma unroll
        for (int r = 0; r < 4; ++r)
          part[e + 1][r] = part[e][r] - __uint_as_float(r & 1 ? packed[r >> 1] & 0xffff0000u : packed[r >> 1] << 16);
      }
#pragma unroll
      for (int e = 0; e < SETS; ++e) {
        const int mine = GQA == 8 ? (e == 0 ? col / GQA : 2) : col / GQA;
        f32x4 x;
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = mine == 0 ? part[0][r] : mine == 1 ? part[1][r] : part[2][r];
        const u32x2 packed = __builtin_bit_cast(u32x2, __builtin_convertvector(x, bf16x4_cvt));
        pf[e].u[tt * 2] = packed[0];
        pf[e].u[tt * 2 + 1] = packed[1];
      }
    }
    hold();
    // ---- P V: dims 16 i.. by 16 columns; lane (col, grp) has the same keys of either operand ----
#pragma unroll
    for (int i0 = 0; i0 < 8; i0 += 4) {
      union { s16x4 half[2]; bf16x8_mfma m; } vf[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
          vf[i].half[tt] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) s16x4*)(uintptr_t)((turn_at ^ ((i0 + i) << 5)) + tt * 4096));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < SETS; ++e)
          o[e][i0 + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[i].m, pf[e].m, o[e][i0 + i], 0, 0, 0);
    }
    hold();
    __builtin_amdgcn_sched_barrier(0);
  };
  if (t < tiles) {
    row = row_of(t, bt[block_of(key_of(t))]);
    block = bt[block_of(key_of(min(t + step, tiles - 1)))];
    asm volatile("" : "+v"(block));        // here, not behind K and V
    __builtin_amdgcn_sched_barrier(0);
    load_k(row, std::true_type());
    __builtin_amdgcn_sched_barrier(0);
    load_v(row);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
    for (; t + step < tiles; t += step) tile(std::true_type());
    tile(std::false_type());
  }

  // ---- fold the lane groups' keys, then the parts and the waves ---------------------------
  const int end_lane = lane_now(), tid = wave * 64 + end_lane;
  l_run += __shfl_xor(l_run, 16);
  l_run += __shfl_xor(l_run, 32);
  float* const sums = reinterpret_cast<float*>(strip);
#pragma unroll
  for (int e = 0; e < SETS; ++e) {
    const int n = e * 16 + (end_lane & 15);  // part n / GQA of head n % GQA
    if constexpr (ONE) {                     // a sum for each set of keys
      f32x4* const to = reinterpret_cast<f32x4*>(sums + (end_lane >> (FP8 ? 3 : 4)) * SUM_PITCH + (end_lane & (FP8 ? 7 : 15)) * DIMS);
#pragma unroll
      for (int i = 0; i < DIMS / 4; ++i) to[i] = o[0][i];
    } else if (n < 3 * GQA) {
#pragma unroll
      for (int i = 0; i < 8; ++i) *reinterpret_cast<f32x4*>(sums + n * SUM_PITCH + i * 16 + (end_lane >> 4) * 4) = o[e][i];
    }
  }
  if (end_lane < GQA) {
    m_lds[wave][end_lane] = m_run;
    l_lds[wave][end_lane] = l_run;
  }
  __syncthreads();
  float* base = partials + (((int64_t)b * num_kv_heads + g_kv) * gridDim.z + z) * GQA * PART_STRIDE;
  // dims of a thread: one round for all of them. (Four of each group size: 0.8 us more without groups)
  constexpr int VEC = GQA > 2 ? GQA / 2 : 1;
  if (tid * VEC < GQA * 128) {
    const int h = tid * VEC >> 7, d = tid * VEC & 127;
    float M = m_lds[0][h];
#pragma unroll
    for (int w = 1; w < 4; ++w) M = fmaxf(M, m_lds[w][h]);
    float acc[VEC] = {}, l = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float e = m_lds[w][h] == -INFINITY ? 0.0f : exp_of<LOCAL>(m_lds[w][h] - M);   // a wave without a tile
      const float* s = reinterpret_cast<const float*>(strips[w]) + h * SUM_PITCH + d;
#pragma unroll
      for (int r = 0; r < VEC; ++r) {
        // an infinite value times what is left of P, which may be 0 or negative, is no number: P's first part alone then.
        // (Asked of the first part itself, the others are read in a branch behind it, 0.4 us a launch)
        if constexpr (ONE) {
          float all = s[0];
#pragma unroll
          for (int i = 1; i < (FP8 ? 8 : 4); ++i) all += s[i * SUM_PITCH];
          acc[r] += all * e;
        } else {
          const float all = s[r] + (s[GQA * SUM_PITCH + r] + s[2 * GQA * SUM_PITCH + r]);
          acc[r] += (all == all ? all : s[r]) * e;
        }
      }
      l += l_lds[w][h] * e;
    }
    if (Z == 1) {
      const float open = head_gate<LOCAL>(gate, gate_stride, b, g_kv * GQA + h);
      short* const to = (short*)out + ((int64_t)b * num_kv_heads * GQA + g_kv * GQA + h) * 128 + d;
#pragma unroll
      for (int r = 0; r < VEC; ++r) to[r] = f32_to_bf16((l > 0.0f ? acc[r] / l : 0.0f) * open);
    } else if (!arrived) {
#pragma unroll
      for (int r = 0; r < VEC; ++r) base[h * PART_STRIDE + d + r] = acc[r];
      if (d == 0) {
        base[h * PART_STRIDE + 128] = M;
        base[h * PART_STRIDE + 129] = l;
      }
    } else {
      const auto far = __builtin_amdgcn_make_buffer_rsrc(base, 0, GQA * PART_STRIDE * 4, 0x00020000);
      const int at = h * PART_STRIDE * 4;
      if constexpr (VEC == 4) {
        const u32x4 all = {__float_as_uint(acc[0]), __float_as_uint(acc[1]), __float_as_uint(acc[2]), __float_as_uint(acc[3])};
        __builtin_amdgcn_raw_buffer_store_b128(all, far, at + d * 4, 0, FAR);
      } else if constexpr (VEC == 2) {
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(acc[0]), __float_as_uint(acc[1])}, far, at + d * 4, 0, FAR);
      } else {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[0]), far, at + d * 4, 0, FAR);
      }
      if (d == 0) __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(M), __float_as_uint(l)}, far, at + 512, 0, FAR);
    }
  }
  if (Z == 1 || !arrived) return;
  // ---- the last workgroup to arrive merges the partials, in their order ----------------------
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  int* const last = reinterpret_cast<int*>(strips[0]);
  if (tid == 0) {
    int* const count = arrived + ((int64_t)b * num_kv_heads + g_kv) * apart;
    *last = __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == Z - 1;
    if (*last) __hip_atomic_store(count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!*last) return;
  // 32 lanes a head, 4 dims each, and as many sets of heads as there are threads for, a partial each in turn; the loads of
  // MERGED partials before the first wait. (Without the sets 16 partials took 0.5 us more)
  constexpr int SETS_OF_HEADS = NTHREADS / (32 * GQA);
  const float* all = base - (int64_t)z * GQA * PART_STRIDE;
  const auto far = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(all), 0, Z * GQA * PART_STRIDE * 4, 0x00020000);
  const int h = (tid >> 5) % GQA, d = (tid & 31) * 4, set = tid / (32 * GQA);
  float M = -INFINITY, sum = 0.0f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int z0 = 0; z0 < Z; z0 += MERGED * SETS_OF_HEADS) {
    f32x4 part[MERGED];
    float m[MERGED], l[MERGED];
#pragma unroll
    for (int e0 = 0; e0 < MERGED; e0 += 4)
      if (z0 + e0 * SETS_OF_HEADS < Z) {
#pragma unroll
        for (int e = e0; e < e0 + 4; ++e) {  // behind the last one zeros
          const int mine = z0 + e * SETS_OF_HEADS + set, at = (mine * GQA + h) * PART_STRIDE * 4;
          const auto ml = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(far, at + 512, 0, FAR));
          part[e] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(far, at + d * 4, 0, FAR));
          m[e] = mine < Z ? ml[0] : -INFINITY;
          l[e] = ml[1];
        }
      }
    const float before = M;
#pragma unroll
    for (int e = 0; e < MERGED; ++e)
      if (z0 + e * SETS_OF_HEADS < Z) M = fmaxf(M, m[e]);
    const float a = before == -INFINITY ? 0.0f : exp_of<LOCAL>(before - M);
    sum *= a;
    acc *= a;
#pragma unroll
    for (int e = 0; e < MERGED; ++e)
      if (z0 + e * SETS_OF_HEADS < Z) {
        const float w = m[e] == -INFINITY ? 0.0f : exp_of<LOCAL>(m[e] - M);
        sum += l[e] * w;
        acc += part[e] * w;
      }
  }
  if constexpr (SETS_OF_HEADS > 1) {       // the sets' sums meet in LDS, behind the one word that said who was last
    f32x4* const sums_of = reinterpret_cast<f32x4*>(strips[1]);
    f32x2* const ml_of = reinterpret_cast<f32x2*>(strips[2]);
    sums_of[tid] = acc;
    ml_of[tid] = f32x2{M, sum};
    __syncthreads();
    if (set > 0) return;
    float top = M;
#pragma unroll
    for (int e = 1; e < SETS_OF_HEADS; ++e) top = fmaxf(top, ml_of[tid + e * 32 * GQA][0]);
    const float a = M == -INFINITY ? 0.0f : exp_of<LOCAL>(M - top);
    sum *= a;
    acc *= a;
#pragma unroll
    for (int e = 1; e < SETS_OF_HEADS; ++e) {
      const f32x2 ml = ml_of[tid + e * 32 * GQA];
      const float w = ml[0] == -INFINITY ? 0.0f : exp_of<LOCAL>(ml[0] - top);
      sum += ml[1] * w;
      acc += sums_of[tid + e * 32 * GQA] * w;
    }
  }
  const float open = head_gate<LOCAL>(gate, gate_stride, b, g_kv * GQA + h);
  bf16x4_vec v;
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = f32_to_bf16((sum > 0.0f ? acc[r] / sum : 0.0f) * open);
  *reinterpret_cast<bf16x4_vec*>((short*)out + ((int64_t)b * num_kv_heads * GQA + g_kv * GQA + h) * 128 + d) = v;
}

template <int GQA, int KV, bool LOCAL>
__global__ __launch_bounds__(NTHREADS, GQA == 8 ? 2 : GQA == 1 && KV != KV_FP8_ANY ? 4 : 3) void attn_decode_tiles(
    float* __restrict__ partials,
    bf16_t* __restrict__ out,            // written where one workgroup has the context, or by the last one with ``arrived``
    const bf16_t* __restrict__ q,        // [B, H, 128], row stride q_tstride
    const char* __restrict__ k_cache,    // [NB, KVH, BS, 128], bf16 or fp8
    const char* __restrict__ v_cache,
    const float* __restrict__ k_scale,   // [NB, KVH, BS] per-row dequant (FP8 only)
    const float* __restrict__ v_scale,
    const int* __restrict__ block_tables,  // [B, max_blocks]
    const int* __restrict__ context_lens,  // [B]
    const bf16_t* __restrict__ gate, int gate_stride,  // [B, H] logits of the heads' sigmoid gates, or nullptr
    int* __restrict__ arrived, int apart,  // [B, KVH] zeros, ``apart`` ints from each other, zeros again afterwards, or nullptr
    float scale, int block_size, uint32_t block_inverse, int max_blocks, int q_tstride, int mask_size, DecodeShares shares, int rows) {
  __shared__ __attribute__((aligned(16))) char strips[4][Strip<GQA>::BYTES];
  __shared__ float m_lds[4][GQA], l_lds[4][GQA];
  const int b = blockIdx.y;
  const bool after = b > 0, ahead = b + 1 < rows;
  int L = context_lens[b];
  bool shared = false;                     // the neighbours' first blocks are this context's: so are more, and lie in the L2
  if constexpr (!LOCAL) {                  // beside the length, not behind it
    const int* bt = block_tables + (int64_t)b * max_blocks;
    int own = bt[0], prev = bt[after ? -max_blocks : 0], next = bt[ahead ? max_blocks : 0];
    asm volatile("" : "+s"(L), "+s"(own), "+s"(prev), "+s"(next));
    shared = (after && prev == own) || (ahead && next == own);
  }
  const int first = first_key(L, mask_size);
  const int tiles = (L - first + TKEYS - 1) / TKEYS;
  const int Z = shares_of(tiles, shares, GQA == 1 && shared);
  if ((int)blockIdx.z >= Z) return;
#define DECODE_SHARE(ONCE)                                                                                                    \
  decode_share<GQA, KV, LOCAL, ONCE>(partials, out, q, k_cache, v_cache, k_scale, v_scale, block_tables, context_lens, gate,   \
                                     gate_stride, arrived, apart, scale, block_size, block_inverse, max_blocks, q_tstride, mask_size, \
                                     shares, L, first, tiles, Z, strips, m_lds, l_lds)
  // both sides whole: with the loops alone twice in one body it spilled registers
  if constexpr (!LOCAL) {
    if (!shared && (int64_t)L * rows * gridDim.x * (KV == KV_BF16 ? 512 : 256) >= DECODE_ONCE) {
      DECODE_SHARE(true);
      return;
    }
  }
  DECODE_SHARE(false);
#undef DECODE_SHARE
}

// Rows of one launch: they lie on the grid's y, which ends at 65535. Steps with a row
// per token (prompt portions on the fp8 cache, short segments) can have more and go out
// in several launches; on x, beside the kv heads, every workgroup would divide.
#define MAX_ROWS 65535

// What is best for contexts of one length is one workgroup a compute unit, 256 in all, or two or three of them on each; in
// between, some units work on one more than others and are waited for. Their number also has to cover contexts of different
// lengths, whose longest has the same number as all: so the longer ones have two or three a unit, in fp8, whose rounds are
// slower, sooner. us by workgroups in all:
//   32 / 8 heads, bf16   one of 7800 168 12.1   248 12.2   488 14.4      5 of 7800 160 31.0   240 30.0   320 35.0   440 30.9   640 32.9
//     16 of 2000 128 27.0   256 25.4   384 27.6   512 25.9   768 26.3      16 / 4, one of 131072 64 90   128 54.8   256 49.4   344 58.9
//     12 of 2500 to 7800 192 50.9   480 47.6      24 of 1300 to 4500 192 61.4   768 53.2      one each, 40 of 2000 64.7, 640 60.5   960 58.4
//   fp8   5 of 7800 240 22.4   320 22.9   440 20.9   640 23.4      16 / 4, 40 of 1500 160 21.1   320 20.3   480 17.8   640 19.6
//     7 of 7000 392 25.3   728 27.2      30 of 600 240 12.2   480 13.5
//   8 / 8   5 of 700 to 7800 240 23.0   440 24.8   fp8 240 19.5   440 16.0 (the lengths of one launch differ: 16.1 with 640 of all)
// Without groups of heads a context whose prompt a neighbour shares is read from the L2, and bound by its rounds: it has two to
// three workgroups a unit at any length (near). 8 / 8 and 16 / 16 heads, us by the rule for the others and so: 11 streams of 1097 12.9,
// 10.2; 7 of 1814 17.5, 13.9; fp8, 15 of 1064 12.0, 10.6; over 65 sizes 4 % less. With groups it gains nothing (4) or little (2).
// Counted over the launch's lengths by each workgroup, so that all are equally long, they took 0.6 us more and gained nothing.
// A merge in its own launch takes 1 us more, but many partials of eight heads take a single workgroup longer. 8 / 1 heads, one
// of 500 7.8, in a launch of its own 8.4; of 7800 12.1, 11.0; of 32768 19.0, 14.5; of 131072 32.1, 22.5: so where tables are long.
static DecodeShares attn_decode_shares(int B, int num_kv_heads, int gqa, int max_ctx, bool fp8, bool local, bool joined) {
  const int64_t pairs = (int64_t)B * num_kv_heads;
  if (gqa == 8 && pairs <= 2 && max_ctx > 16384) joined = false;
  DecodeShares s;
  s.joined = joined;
  s.near = 0;
  if (joined && !local && gqa == 1 && pairs <= 256) {        // of two to three workgroups a unit what fills the units best
    double best = 0.0;
    for (int64_t z = 512 / pairs; z <= 768 / pairs; ++z) {
      const double fill = (double)(pairs * z) / ((pairs * z + 255) / 256 * 256);
      if (fill >= best) best = fill, s.near = (int)z;
    }
  }
  s.few = joined ? 3 : local ? 1 : 2;
  if (pairs <= 256) {
    s.lo = joined ? 32 : 48;
    s.per = joined ? 16 : 4;
    for (int i = 0; i < 3; ++i) {
      s.most[i] = (int)std::min<int64_t>(256 * (i + 1) / pairs, 128);
      s.from[i] = i == 0 ? 0 : std::max(6, (fp8 ? 2 * i : 2 * i + 2) * s.most[i]);
      // not where it fills the units less, nor, in fp8 and with groups, three a unit where it does not fill them better
      const int64_t full = (int64_t)s.most[i] * pairs * i, before = i ? (int64_t)s.most[i - 1] * pairs * (i + 1) : 0;
      const int by = fp8 && gqa > 1 && i == 2 ? -24 * i * (i + 1) : 24 * i * (i + 1);
      if (i && full + by < before) s.most[i] = s.most[i - 1], s.from[i] = INT32_MAX;
    }
  } else {                                   // those that fill whole rounds of the units best, one for every eight rounds
    s.lo = 1;
    s.per = 8;
    s.most[0] = 1;
    s.from[1] = s.from[2] = INT32_MAX;
    double best = 0.0;
    for (int z = 1; z == 1 || pairs * z <= 1024; ++z) {
      if (pairs * z < 512 && fp8 && pairs * (z + 1) <= 1024) continue;
      const double fill = (double)(pairs * z) / ((pairs * z + 255) / 256 * 256);
      if (fill > best + 0.02) best = fill, s.most[0] = z;
    }
  }
  const int rounds = (int)(((int64_t)max_ctx + 4 * TKEYS - 1) / (4 * TKEYS));
  s.grid = rounds <= s.few ? 1 : std::min(most_of(rounds, s, true), rounds);
  return s;
}

// workgroups per context of a launch: room for partials where more than one
extern "C" int attn_decode_splits(int B, int num_kv_heads, int gqa, int max_ctx, int fp8, int local, int joined) {
  return attn_decode_shares(B < MAX_ROWS ? B : MAX_ROWS, num_kv_heads, gqa, max_ctx, fp8 != 0, local != 0, joined != 0).grid;
}

// merge the partials of a (stream, q head): two dims per lane, the partials dealt
// to four waves
template <bool LOCAL>
__global__ void __launch_bounds__(256) attn_decode_merge_kernel(
    bf16_t* __restrict__ out,            // [B, H, 128]
    const float* __restrict__ partials,  // [B, KVH, Z, gqa, 130]
    const int* __restrict__ context_lens, const bf16_t* __restrict__ gate, int gate_stride, int gqa, int Z,
    int mask_size, DecodeShares shares) {
  const int b = blockIdx.y, h = blockIdx.x, num_q_heads = gridDim.x;
  const int g_kv = h / gqa, g = h % gqa;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int L = context_lens[b];
  const int tiles = (L - first_key(L, mask_size) + TKEYS - 1) / TKEYS;
  const int n = shares_of(tiles, shares, false);     // not joined: near is 0
  if (n == 1) return;                    // its one workgroup has written the result
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

// picks the GQA instantiation (the binding admits 1, 2, 4, 8); mask_size: -1 plain decode,
// from 0 on a block-local layer's (bf16 caches); partials: room for
// min(B, MAX_ROWS) * KVH * splits * gqa * 130 floats when splits > 1
extern "C" void launch_attn_decode(
    bf16_t* out, float* partials, int* arrived, int apart, const bf16_t* q, const void* k_cache, const void* v_cache,
    const float* k_scale, const float* v_scale, const int* block_tables, const int* context_lens,
    const bf16_t* gate, int gate_stride, float scale, int num_q_heads, int num_kv_heads, int block_size,
    int max_blocks, int max_ctx, int q_tstride, int B, int cache_fp8, int mask_size, hipStream_t stream) {
  const int gqa = num_q_heads / num_kv_heads;
  const bool local = mask_size >= 0;
  const DecodeShares sh = attn_decode_shares(B < MAX_ROWS ? B : MAX_ROWS, num_kv_heads, gqa, max_ctx, cache_fp8 != 0, local, arrived != nullptr);
  const int splits = sh.grid;
  if (!sh.joined) arrived = nullptr;
  const bool quads = block_size % 4 == 0 && (reinterpret_cast<uintptr_t>(k_scale) | reinterpret_cast<uintptr_t>(v_scale)) % 16 == 0;
  const uint32_t block_inverse = block_size > 1 ? (uint32_t)(((1ull << 32) + block_size - 1) / block_size) : ~0u;
  for (int b0 = 0; b0 < B; b0 += MAX_ROWS) {
    const int rows = B - b0 < MAX_ROWS ? B - b0 : MAX_ROWS;
    const dim3 grid(num_kv_heads, rows, splits);
    bf16_t* o = out + (int64_t)b0 * num_q_heads * 128;
    const bf16_t* q0 = q + (int64_t)b0 * q_tstride;
    const int* bt = block_tables + (int64_t)b0 * max_blocks;
    int* a0 = arrived ? arrived + (int64_t)b0 * num_kv_heads * apart : nullptr;
    const bf16_t* g0 = gate ? gate + (int64_t)b0 * gate_stride : nullptr;
#define LAUNCH(G, F, L)                                                                            \
  hipLaunchKernelGGL((attn_decode_tiles<G, F, L>), grid, dim3(NTHREADS), 0, stream, partials, o, q0, \
                     (const char*)k_cache, (const char*)v_cache, k_scale, v_scale, bt,             \
                     context_lens + b0, g0, gate_stride, a0, apart, scale, block_size, block_inverse, max_blocks, q_tstride, \
                     mask_size, sh, rows)
#define DISPATCH(G) \
  do {                                                                                             \
    if (cache_fp8 && quads) LAUNCH(G, KV_FP8, false);                                              \
    else if (cache_fp8) LAUNCH(G, KV_FP8_ANY, false);                                              \
    else if (local) LAUNCH(G, KV_BF16, true);                                                      \
    else LAUNCH(G, KV_BF16, false);                                                                \
  } while (0)
    switch (gqa) {
      case 1: DISPATCH(1); break;
      case 2: DISPATCH(2); break;
      case 4: DISPATCH(4); break;
      default: DISPATCH(8); break;
    }
#undef DISPATCH
#undef LAUNCH
    if (splits > 1 && !arrived)
      hipLaunchKernelGGL(local && !cache_fp8 ? attn_decode_merge_kernel<true> : attn_decode_merge_kernel<false>,
                         dim3(num_q_heads, rows), dim3(256), 0, stream, o, partials, context_lens + b0, g0,
                         gate_stride, gqa, splits, mask_size, sh);
  }
}
