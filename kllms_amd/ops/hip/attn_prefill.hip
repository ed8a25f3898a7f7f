// Causal prefill attention for gfx950 - flash-style MFMA kernel over rows of packed
// sequences, keys either from the same packed rows or from the paged cache.
//
//   - an 8-wave workgroup serves 8 consecutive 32-row q-tiles of ONE (sequence,
//     q-head); 128 keys at a time are staged in LDS for all waves, double-buffered:
//     the next 128 are on their way there, without registers in between, while these
//     are multiplied, 64 at a time
//   - SWAPPED QK^T: S = mfma(A=K_tile, B=Q), so a lane's accumulators hold one q-row's
//     scores and the softmax is in registers (one permlane32_swap merges the halves)
//   - P goes to bf16 MFMA B-fragments with pack + half swaps; O^T = mfma(A=V^T, B=P).
//     The paged form multiplies P as three bf16 parts, 24 bits: exactly the fp32 P
//     of the decode kernel, which rows behind a cache otherwise take
//     V lies in LDS as it lies in memory; ds_read_b64_tr_b16 turns it on the way to
//     the fragment (staging it transposed took 16 two-byte LDS writes a thread)
//   - K's 16-byte units are XORed with the row, V's 32-byte slots with v_turn of it:
//     both fragment reads are free of bank conflicts
//   - where few segments (the tail of a chat behind a long cache) would leave the chip idle,
//     groups are of 64 rows and four waves share a q-tile, 32 keys of each stage each; their
//     sums meet in LDS
//
// What bounds it: a SIMD's two waves, which a barrier keeps in step, do their 32 matrix
// instructions of a tile (1024 cycles) and their softmax (about 1000 cycles, half of
// them the exponentials at a quarter of the rate) at the same times, so that the two
// add up: 3600 cycles for both, matrix and vector units busy 41 and 43 % each. So the
// barriers are few, the softmax is kept lean - base-2 exponentials of one fma each, the
// mask only where a tile crosses the diagonal or the end, the packed conversion
// instruction, and a running max that is renewed only when it grows by more than 8 (P
// stays below e^8, fine in fp32 and bf16) - and P V has priority over the other wave.
// Taken back: waves in turns, one at its products while the other is at its softmax,
// with barriers between (a turn took 2400 cycles); the next tile's scores ahead of this
// one's softmax (3 % faster for long sequences, 15 % slower for short and paged ones);
// 64 rows a wave, whose sums and scores the registers do not hold.
//
// Grid: q-heads fastest, the heads of a kv head 8 apart, so that with 8 kv heads an
// XCD's L2 serves one of them; groups of rows longest first, since causal groups
// differ in length.
//
// Measured in graphs, 32 heads / 8 kv heads, with 64 keys a stage by way of registers and
// so, us: one sequence of 7777 rows 548, 502 (986 TFLOP/s), 24 of about 550 177, 142; 16 / 4
// heads, 8 of 1000 76, 67; 8 segments of 160 rows behind 1536 cached keys 98, 95, 12 of 45
// behind 2000 135, 85, one of 37 behind 1536 52, 33; in groups of 64 rows where that is faster
// (paged_prefill_few), one of 146 behind 1536 82, 36, of 512 98, 47, four of 146 83, 63.
//
// MFMA fragment maps (v_mfma_f32_32x32x16_bf16, verified on-device by the
// mfma_selftest binding):
//   A[i][k]: lane l holds i = l&31, k = (l>>5)*8 + j   (j = 0..7)
//   B[k][j]: lane l holds j = l&31, k = (l>>5)*8 + jj
//   C/D[i][j]: lane l holds j = l&31, i = (r&3) + 8*(r>>2) + 4*(l>>5)  (r = 0..15)
// ds_read_b64_tr_b16, per 16 lanes: lane 4r + c addresses row r, elements 4c..4c+3 of
// 16; lane i receives element i of rows 0..3.

#include "common.h"

typedef __bf16 bf16x8_mfma __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

#define QBLK 32
#define STAGE 128                  // keys staged per barrier round
#define DHEAD 128
#define NWAVES 8
#define STAGE_BYTES (STAGE * 256)  // K or V of a stage
#define LDS_BYTES (4 * STAGE_BYTES)
#define SHARE_FLOATS (66 * 64)     // sums of a wave, its maxima and row sums

__device__ __forceinline__ int acc_row(int r, int half) {
  return (r & 3) + 8 * (r >> 2) + 4 * half;   // C/D row map
}

// V's 32-byte slots of a row are XORed with this: the rows of a turned read, 4 by 2 slots, lie in all banks
__device__ __forceinline__ int v_turn(int row) { return (row & 3) * 2 + (row >> 2 & 1); }

// SHARED: PAGED, groups of 64 rows: four waves share a q-tile, each with 32 keys of a stage
template <bool PAGED, bool SHARED>
__global__ void __launch_bounds__(64 * NWAVES) attn_prefill_kernel(
    bf16_t* __restrict__ out,       // [T, H, D] contiguous
    const bf16_t* __restrict__ q,   // [T, H, D], token stride q_tstride
    const bf16_t* __restrict__ k,   // [T, KVH, D], token stride kv_tstride; PAGED: cache [NB, KVH, BS, D]
    const bf16_t* __restrict__ v,
    const int* __restrict__ grp_start,   // [G] first row of the group's sequence
    const int* __restrict__ grp_len,     // [G] rows of the sequence, 0: idle group
    const int* __restrict__ grp_q0,      // q0_stride 1: [G] group's first row within the sequence, its waves' 32 rows
                                         // following; 8: [G, 8] first row of each wave, -1: none
    const int* __restrict__ grp_seg,     // PAGED: [G] row of block_tables / seg_pos
    const int* __restrict__ block_tables, const int* __restrict__ seg_pos,  // PAGED: position of a segment's row 0
    float scale, int num_kv_heads, int q_tstride, int kv_tstride, int q0_stride, int block_size, uint32_t block_inverse, int max_blocks) {
  const int grp = blockIdx.y;
  const int num_q_heads = gridDim.x;
  const int g_kv = blockIdx.x % num_kv_heads;
  const int h = g_kv * (num_q_heads / num_kv_heads) + blockIdx.x / num_kv_heads;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int half = lane >> 5;
  const int col = lane & 31;       // q-row (B/C col) or K row / V^T row (A row)

  const int seqlen = grp_len[grp];
  int qrow0, rows_end = 0;         // this wave's first row; behind the group's last one
  constexpr int SHARES = SHARED ? 4 : 1;
  const int share = wave % SHARES;
  if (PAGED || q0_stride == 1) {
    const int q0 = grp_q0[grp];
    if (q0 >= seqlen) return;
    rows_end = min(seqlen, q0 + NWAVES / SHARES * QBLK);
    qrow0 = q0 + wave / SHARES * QBLK;
  } else {
    qrow0 = grp_q0[grp * NWAVES + wave];
#pragma unroll
    for (int w = 0; w < NWAVES; ++w) {
      const int r = grp_q0[grp * NWAVES + w];
      if (r >= 0 && r < seqlen) rows_end = max(rows_end, min(seqlen, r + QBLK));
    }
  }
  if (seqlen <= 0 || rows_end <= 0) return;
  const int seq_start = grp_start[grp];
  const int seg = PAGED ? grp_seg[grp] : 0;
  const int pos0 = PAGED ? seg_pos[seg] : 0;          // keys before the sequence's first row
  const bool active = qrow0 >= 0 && qrow0 < rows_end;
  const int my_pos = pos0 + qrow0 + col;
  // keys visible to the group's last row, and to this wave's
  const int kv_end_grp = pos0 + rows_end;
  const int kv_end_me = active ? pos0 + min(rows_end, qrow0 + QBLK) : 0;

  extern __shared__ __attribute__((aligned(1024))) char smem[];          // [buffer][K | V]

  // ---- Q fragments (B-operand): 8 d-slices of 16 --------------------------
  union QFrag { u32x4 u; bf16x8_mfma m; };
  QFrag q_frag[8];
  {
    const int row = active ? min(qrow0 + col, seqlen - 1) : 0;
    const short* qp = (const short*)q + (int64_t)(seq_start + row) * q_tstride + h * DHEAD + half * 8;
    // a negative scale goes into Q's signs: the max below is taken before scaling
    const uint32_t sign = scale < 0.0f ? 0x80008000u : 0u;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      q_frag[s].u = *reinterpret_cast<const u32x4*>(qp + s * 16);
#pragma unroll
      for (int j = 0; j < 4; ++j) q_frag[s].u[j] ^= sign;
    }
  }
  // scores to base-2 exponents; above zero, so that a masked score stays -inf
  const float c2 = fmaxf(fabsf(scale) * 1.44269504088896340736f, 1e-30f);
  const float THR2 = 8.0f * 1.44269504088896340736f;

  // ---- staging: straight to LDS, a copy has four rows, a wave COPIES of them of K and of V --------
  constexpr int COPIES = STAGE / NWAVES / 4;
  const int* bt = PAGED ? block_tables + (int64_t)seg * max_blocks : nullptr;
  typedef __attribute__((address_space(3))) char* lds_t;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_t)smem;
  const int st_row = wave * (COPIES * 4) + (lane >> 4), st_unit = lane & 15;
  int st_block[COPIES];                            // PAGED: of the stage that is asked for next
  // key / block_size by its reciprocal, which is off by one at most
  auto block_of = [&](int key) {
    const int n = (int)__umulhi((uint32_t)key, block_inverse), rest = key - n * block_size;
    return n - (rest < 0) + (rest >= block_size);
  };
  auto st_key = [&](int kt, int i) { return min(kt + st_row + i * 4, kv_end_grp - 1); };
  auto ask_blocks = [&](int kt) {
    if constexpr (PAGED) {
#pragma unroll
      for (int i = 0; i < COPIES; ++i) st_block[i] = bt[block_of(st_key(kt, i))];
    }
  };
  auto stage = [&](int kt, int buf) {
#pragma unroll
    for (int i = 0; i < COPIES; ++i) {
      const int r = st_row + i * 4, key = st_key(kt, i);
      int64_t row;
      if constexpr (PAGED) row = (((int64_t)st_block[i] * num_kv_heads + g_kv) * block_size + (key - block_of(key) * block_size)) * DHEAD;
      else row = (int64_t)(seq_start + key) * kv_tstride + g_kv * DHEAD;
      const uint32_t to = lds0 + buf * 2 * STAGE_BYTES + (wave * COPIES + i) * 1024;
      const uint64_t ka = (uint64_t)((const short*)k + row + ((st_unit ^ (r & 15)) << 3));
      const uint64_t va = (uint64_t)((const short*)v + row + ((st_unit ^ (v_turn(r) << 1)) << 3));
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(ka), "s"(to) : "memory");
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(va), "s"(to + STAGE_BYTES) : "memory");
    }
  };

  f32x16 o_acc[4] = {};
  float m_run = -INFINITY;
  float l_run = 0.0f;

  constexpr int SUBS = SHARED ? 1 : 2, TILE = SUBS * 32;       // 32-key parts and keys of a wave's tile
  auto tile = [&](int ks, int kt, int buf) {
    const char* k_lds = smem + buf * 2 * STAGE_BYTES + (kt - ks) * 256;
    // ---- QK^T: S[key][qrow], 32 keys each ----------------------------
    f32x16 s_acc[SUBS] = {};
#pragma unroll
    for (int s = 0; s < 8; ++s) {
#pragma unroll
      for (int sub = 0; sub < SUBS; ++sub) {
        const int krow = col + sub * 32;
        const bf16x8_mfma a = *reinterpret_cast<const bf16x8_mfma*>(
            k_lds + krow * 256 + (((s * 2 + half) ^ (krow & 15)) << 4));
        s_acc[sub] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, q_frag[s].m, s_acc[sub], 0, 0, 0);
      }
    }
    if (kt + TILE > pos0 + qrow0 || kt + TILE > kv_end_grp) {
      // rows see keys up to their own position, which also ends the sequence
#pragma unroll
      for (int sub = 0; sub < SUBS; ++sub)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = kt + sub * 32 + acc_row(r, half);
          if (key > my_pos || key >= kv_end_grp) s_acc[sub][r] = -INFINITY;
        }
    }

    // ---- online softmax (row = lane-local) --------------------------------
    float tmax = s_acc[0][0];
#pragma unroll
    for (int sub = 0; sub < SUBS; ++sub)
#pragma unroll
      for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, s_acc[sub][r]);
    {
      auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(tmax), __float_as_uint(tmax), false, false);
      tmax = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1])) * c2;
    }
    // the running max is renewed per row (lane) and only when it grows by more
    // than THR2; the first tile always renews it, a tile without a visible key never
    float alpha = 1.0f;
    if (!(tmax <= m_run + THR2)) {
      const float m_new = fmaxf(m_run, tmax);
      alpha = (m_run == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);
      m_run = m_new;
    }
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[dt][r] *= alpha;
      l_run *= alpha;
    }
    // masked scores: fma(-inf, c2, -m) = -inf, whose exponential is 0
    const float m_use = m_run == -INFINITY ? 0.0f : m_run;
    // 32 keys of P to B-fragment words; paged: also what bf16 leaves of it, twice (the
    // differences are exact)
    constexpr int PARTS = PAGED ? 3 : 1;
    auto expo = [&](int sub, uint32_t (&w)[PARTS][8]) {
#pragma unroll
      for (int pr = 0; pr < 8; ++pr) {
        f32x2 p;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s_acc[sub][2 * pr + e], c2, -m_use));
          l_run += p[e];
        }
#pragma unroll
        for (int part = 0; part < PARTS; ++part) {
          w[part][pr] = __builtin_bit_cast(uint32_t, __builtin_convertvector(p, bf16x2_t));
          p[0] -= __uint_as_float(w[part][pr] << 16);
          p[1] -= __uint_as_float(w[part][pr] & 0xffff0000u);
        }
      }
    };

    // ---- PV: O^T += V^T x P, 16 keys at a time ------------------------------
    const char* v_lds = k_lds + STAGE_BYTES;
    // this lane's share of a transposed read: row (lane & 15) / 4, 4 elements
    const int tr_row = half * 8 + ((lane & 15) >> 2);
    const int tr_byte = (lane & 3) * 8;
    const int tr_slot = (lane >> 4) & 1;
    union PFrag { uint32_t w[4]; bf16x8_mfma m; };
    auto fragment = [&](const uint32_t (&packs)[8], int kw) {
      PFrag pf;
      auto r0 = __builtin_amdgcn_permlane32_swap(packs[4 * kw + 0], packs[4 * kw + 2], false, false);
      auto r1 = __builtin_amdgcn_permlane32_swap(packs[4 * kw + 1], packs[4 * kw + 3], false, false);
      pf.w[0] = r0[0];
      pf.w[1] = r1[0];
      pf.w[2] = r0[1];
      pf.w[3] = r1[1];
      return pf;
    };
    auto weighted = [&](int sub, const uint32_t (&w)[PARTS][8]) {
#pragma unroll
      for (int kw = 0; kw < 2; ++kw) {
        PFrag pf[PARTS];
#pragma unroll
        for (int part = 0; part < PARTS; ++part) pf[part] = fragment(w[part], kw);
        const int key = sub * 32 + kw * 16 + tr_row;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
          union { s16x4 t[2]; bf16x8_mfma m; } vf;
#pragma unroll
          for (int rd = 0; rd < 2; ++rd) {
            const int kr = key + rd * 4;
            const char* p = v_lds + kr * 256 + (((dt * 2 + tr_slot) ^ v_turn(kr)) << 5) + tr_byte;
            vf.t[rd] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
          }
#pragma unroll
          for (int part = 0; part < PARTS; ++part)
            o_acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf.m, pf[part].m, o_acc[dt], 0, 0, 0);
        }
      }
    };
    uint32_t pw[SUBS][PARTS][8];
    if constexpr (PAGED) {       // one half after the other: the registers of all six parts are not there
#pragma unroll
      for (int sub = 0; sub < SUBS; ++sub) {
        expo(sub, pw[sub]);
        weighted(sub, pw[sub]);
      }
    } else {
#pragma unroll
      for (int sub = 0; sub < SUBS; ++sub) expo(sub, pw[sub]);
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int sub = 0; sub < SUBS; ++sub) weighted(sub, pw[sub]);
      __builtin_amdgcn_s_setprio(0);
    }
  };
  ask_blocks(0);
  stage(0, 0);
  ask_blocks(STAGE);
  int buf = 0;
  for (int ks = 0; ks < kv_end_grp; ks += STAGE, buf ^= 1) {
    // this stage is there, and the last one's buffer, whose reads have come back, is free
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (ks + STAGE < kv_end_grp) {
      stage(ks + STAGE, buf ^ 1);
      ask_blocks(ks + 2 * STAGE);
    }
    const int end = min(ks + STAGE, kv_end_me);
#pragma unroll 1
    for (int kt = ks + share * TILE; kt < end; kt += SHARES * TILE) tile(ks, kt, buf);
  }

  // ---- the shares' sums, lane by lane, to the first of a q-tile's waves ----------
  if constexpr (SHARED) {
    __syncthreads();
    // of both q-tiles the other three: 6 of 16.5 KB
    float* const sums = reinterpret_cast<float*>(smem) + (wave - wave / SHARES - (share > 0)) * SHARE_FLOATS + lane;
    if (share > 0) {
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) sums[(dt * 16 + r) * 64] = o_acc[dt][r];
      sums[64 * 64] = m_run;
      sums[65 * 64] = l_run;
    }
    __syncthreads();
    if (share > 0) return;
    for (int e = 0; e < SHARES - 1; ++e) {
      const float* theirs = sums + e * SHARE_FLOATS;
      const float m = theirs[64 * 64], m_new = fmaxf(m_run, m);
      const float a = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);
      const float w = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - m_new);
      m_run = m_new;
      l_run = l_run * a + theirs[65 * 64] * w;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[dt][r] = o_acc[dt][r] * a + theirs[(dt * 16 + r) * 64] * w;
    }
  }

  // ---- epilogue: merge half-sums, normalize, write O ----------------------
  {
    auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_run), __float_as_uint(l_run), false, false);
    l_run = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
  }
  if (active && qrow0 + col < rows_end) {
    const float inv_l = (l_run > 0.0f) ? 1.0f / l_run : 0.0f;
    bf16_t* op = out + (((int64_t)(seq_start + qrow0 + col)) * num_q_heads + h) * DHEAD;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
#pragma unroll
      for (int g2 = 0; g2 < 4; ++g2) {   // regs 4*g2..+3 = d consecutive
        const int d0 = dt * 32 + 8 * g2 + 4 * half;
        bf16x4_vec o;
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = f32_to_bf16(o_acc[dt][4 * g2 + j] * inv_l);
        *reinterpret_cast<bf16x4_vec*>((short*)op + d0) = o;
      }
    }
  }
}

// groups of a launch: they lie on the grid's y, which ends at 65535 (a sequence has one at
// least, so many short prompts have as many)
#define MAX_GROUPS 65535

// room for the kernels' LDS; asked for at each launch: the attribute is the current device's
static bool prefill_lds_ready(const void* kernel) {
  return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES) == hipSuccess;
}

// 0, or -1 where the LDS cannot be had
extern "C" int launch_attn_prefill(bf16_t* out, const bf16_t* q, const bf16_t* k, const bf16_t* v,
                                   const int* grp_start, const int* grp_len, const int* grp_q0, int q0_stride,
                                   int ngroups, float scale, int num_q_heads, int num_kv_heads, int q_tstride,
                                   int kv_tstride, hipStream_t stream) {
  if (!prefill_lds_ready(reinterpret_cast<const void*>(attn_prefill_kernel<false, false>))) return -1;
  for (int g = 0; g < ngroups; g += MAX_GROUPS)
    hipLaunchKernelGGL((attn_prefill_kernel<false, false>), dim3(num_q_heads, ngroups - g < MAX_GROUPS ? ngroups - g : MAX_GROUPS),
                       dim3(64 * NWAVES), LDS_BYTES, stream, out, q, k, v, grp_start + g, grp_len + g,
                       grp_q0 + (int64_t)g * q0_stride, nullptr, nullptr, nullptr, scale, num_kv_heads, q_tstride,
                       kv_tstride, q0_stride, 1, ~0u, 0);
  return 0;
}

// rows: of a group, 64 or 256
extern "C" int launch_attn_prefill_paged(bf16_t* out, const bf16_t* q, const bf16_t* k_cache, const bf16_t* v_cache,
                                         const int* grp_start, const int* grp_len, const int* grp_q0,
                                         const int* grp_seg, const int* block_tables, const int* seg_pos, int ngroups,
                                         float scale, int num_q_heads, int num_kv_heads, int q_tstride,
                                         int block_size, int max_blocks, int rows, hipStream_t stream) {
  const auto kernel = rows == 64 ? attn_prefill_kernel<true, true> : attn_prefill_kernel<true, false>;
  if (!prefill_lds_ready(reinterpret_cast<const void*>(kernel))) return -1;
  const uint32_t inverse = block_size > 1 ? (uint32_t)(((1ull << 32) + block_size - 1) / block_size) : ~0u;
  for (int g = 0; g < ngroups; g += MAX_GROUPS)
    hipLaunchKernelGGL(kernel, dim3(num_q_heads, ngroups - g < MAX_GROUPS ? ngroups - g : MAX_GROUPS),
                       dim3(64 * NWAVES), LDS_BYTES, stream, out, q, k_cache, v_cache, grp_start + g, grp_len + g, grp_q0 + g,
                       grp_seg + g, block_tables, seg_pos, scale, num_kv_heads, q_tstride, 0, 1, block_size, inverse,
                       max_blocks);
  return 0;
}

// Groups of 256 rows of each sequence cu[i]..cu[i+1], into plan [3, G] (start, length,
// first row), written back to front - a sequence's last rows see the most keys - and
// idle in front. One workgroup, no host round trip.
__global__ void __launch_bounds__(1024) attn_prefill_plan_kernel(int* __restrict__ plan, const int* __restrict__ cu,
                                                                 int n, int G) {
  __shared__ int sums[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int before = 0;                       // groups of the sequences handled so far
  for (int s0 = 0; s0 < n; s0 += 1024) {
    const int s = s0 + tid;
    const int start = s < n ? cu[s] : 0;
    const int len = s < n ? max(0, cu[s + 1] - start) : 0;
    const int mine = (len + NWAVES * QBLK - 1) / (NWAVES * QBLK);
    int incl = mine;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(incl, off);
      if (lane >= off) incl += o;
    }
    __syncthreads();
    if (lane == 63) sums[wave] = incl;
    __syncthreads();
    int at = before + incl - mine, all = 0;
    for (int w = 0; w < 16; ++w) {
      if (w < wave) at += sums[w];
      all += sums[w];
    }
    for (int j = 0; j < mine; ++j) {
      const int g = G - 1 - (at + j);
      if (g < 0) break;                 // more groups than rows allow: cu is not what the caller said
      plan[g] = start;
      plan[G + g] = len;
      plan[2 * G + g] = j * NWAVES * QBLK;
    }
    before += all;
  }
  for (int g = tid; g < G - before; g += 1024) plan[G + g] = 0;
}

extern "C" void launch_attn_prefill_plan(int* plan, const int* cu, int n, int G, hipStream_t stream) {
  hipLaunchKernelGGL(attn_prefill_plan_kernel, dim3(1), dim3(1024), 0, stream, plan, cu, n, G);
}
