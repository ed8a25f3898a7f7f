// Grouped mixture-of-experts products for gfx950 (prefill shapes):
//
//   moe_sort      (token, choice) pairs grouped by expert, without the host
//   moe_gateup    act[s, :] = silu(x[tok(s)] Wg[e]^T) * (x[tok(s)] Wu[e]^T)
//   moe_down      y[s, :]   = act[s] Wd[e]^T
//   moe_combine   out[t, :] = sum over choices j of w[t, j] y[pos(t, j)], in fp32
//
// The products: a 512-thread workgroup (8 waves, 2 x 4) computes 256 rows of one
// expert by 256 columns (gate/up: 128 gate and the same 128 up columns), 128 x 64 a
// wave with v_mfma_f32_32x32x16_bf16 (fragment maps verified by mfma_selftest.hip).
// K goes by 64 through double-buffered LDS (128 KB, one workgroup per compute unit):
// the next 64 are fetched to registers under the matrix work of these (32 matrix
// instructions a wave and stage, 2048 cycles for the two waves of a SIMD) and written
// to the other buffer between the last ones, one barrier per stage. A stage is one
// branch-free scheduling region whose issue order is fixed: the next k-window's LDS
// reads between this one's matrix instructions (left to itself the compiler reads,
// waits and multiplies in turn: 15% slower). Rows of 128 bytes, their 16-byte units
// XORed with the row: staging and fragment reads are conflict-free.
//
// Why this tile: 128 x 64 a wave reads 6 KB of LDS for 8 matrix instructions, which
// with the staging keeps LDS just below the matrix units; 32 x (64 + 64), the tile this
// replaces, read 5 KB for 4, had one stage of 512 cycles to hide a fetch under, and
// looped over an expert's rows. 256 rows leave padding (about 512 rows an expert at
// 2048 tokens are two or three tiles), so the upper four waves of a tile with at most
// 128 rows only help staging: such a tile takes half the matrix time.
//
// Workgroups are numbered (expert, column tile, row tile), rows fastest, and dealt to
// the 8 XCDs in equal runs: an XCD's L2 sees each weight panel once, for its two or
// three row tiles, and mostly one expert's rows.
//
// Measured at 2048 rows, 8 experts of 14336, top 2, width 4096: gate/up 1198 us (803
// TFLOP/s; 2714 before), down 783 (614: 320 tiles are a round and a quarter; 1347
// before); with routing around them 1.93 - 2.0 ms (4.36). The one tile serves every row
// count: the layer at 65 / 128 / 300 / 512 / 1024 rows takes 765 / 771 / 796 / 856 / 1050 us,
// with 32-row waves over 128-row padding and the routing on the host it took 1195 / 1205 /
// 1177 / 1751 / 2577; with experts of 3584 and 65 rows 253 (623).

#include "common.h"

#define MOE_BM 256
#define MOE_BK 64                      // k-depth per stage (128 B per row)
#define MOE_LDS (2 * 2 * MOE_BM * 128) // two buffers of 256 A rows and 256 B rows

typedef __bf16 bf16x8_mfma __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// byte offset inside a staged tile of 128-byte rows, with the bank-conflict XOR
__device__ __forceinline__ int tile_off(int row, int unit) {
  return row * 128 + ((unit ^ (row & 7)) << 4);
}

// GATEUP: a = x [T, K] gathered by ids, w [E, 2 * N, K] (gate at [0, N), up behind),
// out [S, N]. Down: a = act [S, K], w [E, N, K], out [S, N]. offsets [E + 1]: row range
// of each expert in sorted space.
template <bool GATEUP>
__global__ void __launch_bounds__(512) moe_product_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ a, const bf16_t* __restrict__ w,
    const int* __restrict__ ids,         // GATEUP: [S] token index, or -1 (a zero row)
    const bf16_t* __restrict__ zeros,    // GATEUP: [K]
    const int* __restrict__ offsets, int E, int N, int K) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;   // waves w and w + 4 share a SIMD
  const int half = lane >> 5, col = lane & 31;
  constexpr int BN = GATEUP ? 128 : 256;     // output columns of a workgroup
  const int n_tiles = (N + BN - 1) / BN;

  // ---- which (expert, column tile, row tile): equal runs per XCD -----------
  int total = 0;
  for (int e = 0; e < E; ++e) total += (offsets[e + 1] - offsets[e] + MOE_BM - 1) / MOE_BM;
  total *= n_tiles;
  const int run = (total + 7) / 8;
  int id = (blockIdx.x & 7) * run + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= run || id >= total) return;
  int e = 0, m_begin = 0, m_end = 0, m_tiles = 0;
  for (; e < E; ++e) {
    m_begin = offsets[e];
    m_end = offsets[e + 1];
    m_tiles = (m_end - m_begin + MOE_BM - 1) / MOE_BM;
    if (id < m_tiles * n_tiles) break;
    id -= m_tiles * n_tiles;
  }
  if (e >= E) return;
  const int n0 = (id / m_tiles) * BN;
  const int m0 = m_begin + (id % m_tiles) * MOE_BM;

  // ---- staging: 4 rows of A and of B per thread, 16 bytes each --------------
  const int st_row = tid >> 3, st_unit = tid & 7;   // rows st_row + 64 i
  const char* a_src[4];
  const char* b_src[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = min(m0 + st_row + 64 * i, m_end - 1);
    if constexpr (GATEUP) {
      const int tok = ids[r];
      a_src[i] = (const char*)(tok >= 0 ? a + (int64_t)tok * K : zeros) + st_unit * 16;
      // B rows 0..127 gate, 128..255 up of the same columns
      const int n = min(n0 + ((st_row + 64 * i) & 127), N - 1) + (i >= 2 ? N : 0);
      b_src[i] = (const char*)(w + ((int64_t)e * 2 * N + n) * K) + st_unit * 16;
    } else {
      a_src[i] = (const char*)(a + (int64_t)r * K) + st_unit * 16;
      b_src[i] = (const char*)(w + ((int64_t)e * N + min(n0 + st_row + 64 * i, N - 1)) * K) + st_unit * 16;
    }
  }
  u32x4 ra[4], rb[4];
  auto load = [&](int stage) {
#pragma unroll
    for (int i = 0; i < 4; ++i) ra[i] = *reinterpret_cast<const u32x4*>(a_src[i] + (int64_t)stage * 128);
#pragma unroll
    for (int i = 0; i < 4; ++i) rb[i] = *reinterpret_cast<const u32x4*>(b_src[i] + (int64_t)stage * 128);
  };
  auto store = [&](int buf) {
    char* base = smem + buf * (2 * MOE_BM * 128);
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4*>(base + tile_off(st_row + 64 * i, st_unit)) = ra[i];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<u32x4*>(base + MOE_BM * 128 + tile_off(st_row + 64 * i, st_unit)) = rb[i];
  };

  f32x16 acc[4][2] = {};
  const bool busy = m0 + wm * 128 < m_end;
  // Fragment addresses: rows of a wave's sets differ by multiples of 32, so one XORed
  // offset per k-window serves them all and the rows are immediate offsets.
  int at_kw[4];
#pragma unroll
  for (int kw = 0; kw < 4; ++kw) at_kw[kw] = col * 128 + (((kw * 2 + half) ^ (col & 7)) << 4);
  const int a_off = wm * 128 * 128;
  const int b_off = MOE_BM * 128 + (GATEUP ? wn * 32 : wn * 64) * 128;
  constexpr int B_SET = (GATEUP ? 128 : 32) * 128;   // from a wave's first column set to its second
  const int stages = K / MOE_BK;
  load(0);
  store(0);
  __syncthreads();
  // the last stage fetches and stores itself again: one scheduling region, no branches
  for (int s = 0; s < stages; ++s) {
    load(min(s + 1, stages - 1));
    if (busy) {
      const char* base = smem + (s & 1) * (2 * MOE_BM * 128);
      bf16x8_mfma af[2][4], bf[2][2];
      auto fetch = [&](int kw) {
        const char* p = base + at_kw[kw];
#pragma unroll
        for (int j = 0; j < 2; ++j)
          bf[kw & 1][j] = *reinterpret_cast<const bf16x8_mfma*>(p + b_off + j * B_SET);
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
          af[kw & 1][mt] = *reinterpret_cast<const bf16x8_mfma*>(p + a_off + mt * 32 * 128);
      };
      // the next window's fragments are read under this one's matrix work
      fetch(0);
#pragma unroll
      for (int kw = 0; kw < 4; ++kw) {            // 4 k-windows of 16
        if (kw < 3) fetch(kw + 1);
        else store((s + 1) & 1);
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            acc[mt][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[kw & 1][mt], bf[kw & 1][j], acc[mt][j], 0, 0, 0);
      }
      // order of issue: six reads, then per window the next one's reads between matrix instructions
      __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
#pragma unroll
      for (int kw = 0; kw < 3; ++kw) {
#pragma unroll
        for (int i = 0; i < 6; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
      }
    } else {
      store((s + 1) & 1);
    }
    __syncthreads();
  }

  // lane: column col of the set, rows (r & 3) + 8 (r >> 2) + 4 half of each 32
  if (!busy) return;
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = m0 + wm * 128 + mt * 32 + (r & 3) + 8 * (r >> 2) + 4 * half;
      if (row >= m_end) continue;
      if constexpr (GATEUP) {
        const int n = n0 + wn * 32 + col;
        const float g = acc[mt][0][r];
        if (n < N) ((short*)out)[(int64_t)row * N + n] = f32_to_bf16(g / (1.0f + __expf(-g)) * acc[mt][1][r]);
      } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int n = n0 + wn * 64 + j * 32 + col;
          if (n < N) ((short*)out)[(int64_t)row * N + n] = f32_to_bf16(acc[mt][j][r]);
        }
      }
    }
  }
}

// topi [P] (P = tokens x choices) -> offsets [E + 1], pos [P] = sorted place of each
// pair, ids [P] = token of each sorted place. One workgroup: counts by wave ballots,
// which also give the places (same order as the pairs' within a wave's 64; the order
// inside an expert matters to nobody).
__global__ void __launch_bounds__(1024) moe_sort_kernel(int* __restrict__ ids, int* __restrict__ pos,
                                                        int* __restrict__ offsets, const int64_t* __restrict__ topi,
                                                        int P, int k, int E) {
  extern __shared__ int cnt[];           // [E] counts, then cursors
  const int tid = threadIdx.x, lane = tid & 63;
  for (int e = tid; e < E; e += 1024) cnt[e] = 0;
  __syncthreads();
  for (int p0 = 0; p0 < P; p0 += 1024) {
    const int p = p0 + tid;
    const int e = p < P ? (int)topi[p] : -1;
    for (int c = 0; c < E; ++c) {
      const unsigned long long m = __ballot(e == c);
      if (m && lane == 0) atomicAdd(&cnt[c], (int)__popcll(m));
    }
  }
  __syncthreads();
  if (tid == 0) {
    int at = 0;
    for (int e = 0; e < E; ++e) {
      const int n = cnt[e];
      offsets[e] = at;
      cnt[e] = at;
      at += n;
    }
    offsets[E] = at;
  }
  __syncthreads();
  for (int p0 = 0; p0 < P; p0 += 1024) {
    const int p = p0 + tid;
    const int e = p < P ? (int)topi[p] : -1;
    int place = -1;
    for (int c = 0; c < E; ++c) {
      const unsigned long long m = __ballot(e == c);
      if (!m) continue;
      int first = 0;
      if (lane == 0) first = atomicAdd(&cnt[c], (int)__popcll(m));
      first = __shfl(first, 0);
      if (e == c) place = first + (int)__popcll(m & ((1ULL << lane) - 1));
    }
    if (p < P) {
      pos[p] = place;
      if (place >= 0) ids[place] = p / k;
    }
  }
}

// tokens on the grid's x: y and z stop at 65535, a packed prompt batch does not
__global__ void __launch_bounds__(256) moe_combine_kernel(bf16_t* __restrict__ out, const bf16_t* __restrict__ y,
                                                          const float* __restrict__ weights,
                                                          const int* __restrict__ pos, int k, int nvec) {
  const int t = blockIdx.x;
  const int i = blockIdx.y * 256 + threadIdx.x;
  if (i >= nvec) return;
  float s[8] = {};
  for (int j = 0; j < k; ++j) {
    const int p = pos[(int64_t)t * k + j];
    if (p < 0) continue;
    const float w = weights[(int64_t)t * k + j];
    const bf16x8_vec v = reinterpret_cast<const bf16x8_vec*>(y)[(int64_t)p * nvec + i];
#pragma unroll
    for (int c = 0; c < 8; ++c) s[c] += w * bf16_to_f32(v[c]);
  }
  bf16x8_vec o;
#pragma unroll
  for (int c = 0; c < 8; ++c) o[c] = f32_to_bf16(s[c]);
  reinterpret_cast<bf16x8_vec*>(out)[(int64_t)t * nvec + i] = o;
}

// room for 128 KB of LDS, asked for at each launch: the attribute is the current device's
template <bool GATEUP>
static bool lds_ready() {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(moe_product_kernel<GATEUP>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, MOE_LDS) == hipSuccess;
}

// rows S in sorted space; the grid holds the most tiles that S rows of E experts can
// make. Returns 0, or -1 where the LDS cannot be had
extern "C" int launch_moe_gateup(void* act, const void* x, const void* w, const int* sorted_ids, const int* offsets,
                                 const void* zeros, int S, int E, int IN, int K, hipStream_t stream) {
  if (!lds_ready<true>()) return -1;
  const int64_t blocks = (int64_t)(S / MOE_BM + E) * ((IN + 127) / 128);
  hipLaunchKernelGGL(moe_product_kernel<true>, dim3((blocks + 7) / 8 * 8), dim3(512), MOE_LDS, stream, (bf16_t*)act,
                     (const bf16_t*)x, (const bf16_t*)w, sorted_ids, (const bf16_t*)zeros, offsets, E, IN, K);
  return 0;
}

extern "C" int launch_moe_down(void* y, const void* act, const void* w, const int* offsets, int S, int E, int H,
                               int IN, hipStream_t stream) {
  if (!lds_ready<false>()) return -1;
  const int64_t blocks = (int64_t)(S / MOE_BM + E) * ((H + 255) / 256);
  hipLaunchKernelGGL(moe_product_kernel<false>, dim3((blocks + 7) / 8 * 8), dim3(512), MOE_LDS, stream, (bf16_t*)y,
                     (const bf16_t*)act, (const bf16_t*)w, nullptr, nullptr, offsets, E, H, IN);
  return 0;
}

extern "C" void launch_moe_sort(int* ids, int* pos, int* offsets, const int64_t* topi, int P, int k, int E,
                                hipStream_t stream) {
  hipLaunchKernelGGL(moe_sort_kernel, dim3(1), dim3(1024), E * sizeof(int), stream, ids, pos, offsets, topi, P, k, E);
}

extern "C" void launch_moe_combine(void* out, const void* y, const float* weights, const int* pos, int T, int k,
                                   int H, hipStream_t stream) {
  const int nvec = H / 8;
  hipLaunchKernelGGL(moe_combine_kernel, dim3(T, (nvec + 255) / 256), dim3(256), 0, stream, (bf16_t*)out,
                     (const bf16_t*)y, weights, pos, k, nvec);
}
