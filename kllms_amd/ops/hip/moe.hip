// Grouped mixture-of-experts products for gfx950 (prefill shapes):
//
//   moe_sort      (token, choice) pairs grouped by expert, without the host
//   moe_gateup    act[s, :] = silu(x[tok(s)] Wg[e]^T) * (x[tok(s)] Wu[e]^T)
//   moe_down      y[s, :]   = act[s] Wd[e]^T
//   moe_combine   out[t, :] = sum over choices j of w[t, j] y[pos(t, j)], in fp32
//
// The products run on the 256-column tiles of tile_product.h: a workgroup computes up to 256
// rows of one expert by 256 columns (gate/up: 128 gate and the same 128 up columns, 64 of each a wave).
//
// What bounds them: with a few hundred rows an expert or fewer, the stream of W from memory;
// above, the matrix units. So the row tiles of an expert are even parts of its rows, in
// tiles of 64, 128, 160, 192 or 256 rows: they keep step, and the 2 or 3 of a column run side
// by side on one XCD, whose L2 then sees a panel of W once. (256 rows a tile and a small one
// for the rest: the small ones run ahead, and read W again: at 1024 rows gate/up 603 us
// instead of 525.) Column tiles go to the 8 XCDs in turn, which gives each the same share of
// every expert. Down: the last round of tiles is shared out over K where it would leave half
// of the units idle (with 300 rows 194 us, 251 without).
//
// Measured, 8 experts, top 2, us of gate/up and down, beside 256 x 256 tiles of eight waves that were
// staged through registers:
//   width 4096, experts of 14336   300 rows  356 + 184 (406 + 328)    1024 rows  551 + 343 (730 + 406)
//                                 2048 rows  896 + 471 (1175 + 812)
//   width 4096, experts of 7168   6000 rows  1117 + 566: 1260 TFLOP/s (1394 + 847)
// The layer with its routing at 65 / 150 / 300 / 600 / 1024 / 2048 / 6000 rows, experts of 14336: 582 / 582 / 605 /
// 666 / 949 / 1431 / 3623 us (741 / 760 / 787 / 907 / 1131 / 1935 / 4622).

#include "tile_product.h"

// one tile; GATEUP: a = x [T, K] gathered by ids, w [E, 2 * N, K] (gate at [0, N), up behind), out [S, N].
// Down: a = act [S, K], w [E, N, K], out [S, N]
template <bool GATEUP, int MJ>
__device__ __forceinline__ void moe_tile(bf16_t* __restrict__ out, const bf16_t* __restrict__ a,
                                         const bf16_t* __restrict__ w, const int* __restrict__ ids,
                                         const bf16_t* __restrict__ zeros, int e, int m0, int m_end, int n0, int N,
                                         int K, const TileShare& sh, char* smem) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  f32x4 acc[8][MJ];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int m = m0 + (wave & 1) * MJ * 16;         // first row of this wave's results
  const int stages = sh.length(K / TP_K);
  const int64_t k0 = (int64_t)sh.first(K / TP_K) * TP_K;
  if constexpr (GATEUP) {
    // W rows of a tile: 64 gate, 64 up, the next 64 gate, 64 up
    const int n_put = n0 + (wave >> 1) * 64;
    const TileRows wr(w + ((int64_t)e * 2 + (wave & 1)) * N * K + k0, n_put, N, 64, K, lane);
    TileGather<MJ> xr;
#pragma unroll
    for (int i = 0; i < MJ; ++i) {
      const int r = min(m0 + wave * MJ * 8 + i * 8 + (lane >> 3), m_end - 1);
      const int tok = ids[r];
      xr.at[i] = (uint64_t)(tok >= 0 ? a + (int64_t)tok * K : zeros) + k0 * 2 + (((lane & 7) ^ (lane >> 3)) << 4);
    }
    tile_product<MJ>(acc, wr, xr, stages, stages * (blockIdx.x & 7) / 8, smem);
    const int n = n0 + (wave >> 1) * 64;
    tile_store<4, MJ>(out + (int64_t)m * N + n, N, m_end - m, N - n, smem, [&](int i, int j) {
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float g = acc[i][j][r];
        v[r] = g / (1.0f + __expf(-g)) * acc[i + 4][j][r];
      }
      return tp_pack(v[0], v[1], v[2], v[3]);
    });
  } else {
    const int n_put = n0 + wave * 64, m_put = m0 + wave * MJ * 8;
    const TileRows wr(w + (int64_t)e * N * K + k0, n_put, N, 64, K, lane);
    const TileRows xr(a + k0, m_put, m_end, MJ * 8, K, lane);
    tile_product<MJ>(acc, wr, xr, stages, stages * (blockIdx.x & 7) / 8, smem);
    if (sh.shares > 1 && !tile_fold<MJ>(acc, sh.part, sh.share, sh.shares, sh.count, smem)) return;
    const int n = n0 + (wave >> 1) * 128;
    tile_store<8, MJ>(out + (int64_t)m * N + n, N, m_end - m, N - n, smem,
                      [&](int i, int j) { return tp_pack(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]); });
  }
}

// offsets [E + 1]: row range of each expert in sorted space; ids [S]: token index of a
// sorted row, or -1 (a row of zeros, [K]). Down: part, count: room for the shares of
// tiles, or nullptr: every tile is one workgroup's.
template <bool GATEUP>
__global__ void __launch_bounds__(TP_THREADS, 1) moe_product_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ a, const bf16_t* __restrict__ w,
    const int* __restrict__ ids, const bf16_t* __restrict__ zeros, const int* __restrict__ offsets,
    float* __restrict__ part, int* __restrict__ count, int E, int N, int K) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  constexpr int BN = GATEUP ? 128 : 256;           // output columns of a workgroup
  const int n_tiles = (N + BN - 1) / BN;
  // (expert, column tile) pairs in turn to the XCDs, the row tiles of one behind each other
  const int xcd = blockIdx.x & 7, lane = threadIdx.x & 63;
  auto first_of = [&](int e) { return (xcd + 8 - (int)((int64_t)e * n_tiles & 7)) & 7; };   // this XCD's first column tile of e
  // its tiles of expert e; a lane each: an expert after the other, 128 of them took 25 us a walk
  auto tiles_of = [&](int e) {
    if (e >= E) return 0;
    const int first = first_of(e);
    return (first < n_tiles ? (n_tiles - first + 7) / 8 : 0) * ((offsets[e + 1] - offsets[e] + 255) / 256);
  };
  auto before_and = [&](int n) {                   // over the wave: the sum up to and with this lane
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(n, off);
      if (lane >= off) n += o;
    }
    return n;
  };
  int tiles = 0;
  if (part)
    for (int e0 = 0; e0 < E; e0 += 64) tiles += __builtin_amdgcn_readlane(before_and(tiles_of(e0 + lane)), 63);
  const TileShare sh(blockIdx.x >> 3, tiles, K / TP_K, part, count, xcd);
  int at = sh.tile, e = E;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int mine = tiles_of(e0 + lane), sum = before_and(mine), all = __builtin_amdgcn_readlane(sum, 63);
    if (at >= all) {
      at -= all;
      continue;
    }
    const int found = (int)__builtin_ctzll(__ballot(at < sum));
    e = e0 + found;
    at -= __builtin_amdgcn_readlane(sum - mine, found);
    break;
  }
  if (e >= E) return;
  const int begin = offsets[e], end = offsets[e + 1], m_tiles = (end - begin + 255) / 256, first = first_of(e);
  // an expert's rows in even parts: its row tiles keep step, and read W from memory once
  const int rows = (end - begin + m_tiles - 1) / m_tiles;
  const int n0 = (first + at / m_tiles * 8) * BN, m0 = begin + at % m_tiles * rows, m_end = min(end, m0 + rows);
#define MOE_TILE(MJ) moe_tile<GATEUP, MJ>(out, a, w, ids, zeros, e, m0, m_end, n0, N, K, sh, smem)
  if (rows > 192) MOE_TILE(8);
  else if (rows > 160) MOE_TILE(6);
  else if (rows > 128) MOE_TILE(5);
  else if (rows > 64) MOE_TILE(4);
  else MOE_TILE(2);
#undef MOE_TILE
}

// topi [P] (P = tokens x choices) -> offsets [E + 1], pos [P] = sorted place of each
// pair, ids [P] = token of each sorted place, an expert's in the order of the pairs: which
// of the products' tiles a row falls into, and with it the order of its sums, is so the
// same in every call. One workgroup, a run of the pairs to each of its ``waves`` waves
// that count: by ballots, which also give the places, in a row of counts of its own.
#define SORT_WAVES 16

__global__ void __launch_bounds__(64 * SORT_WAVES) moe_sort_kernel(int* __restrict__ ids, int* __restrict__ pos,
                                                                   int* __restrict__ offsets,
                                                                   const int64_t* __restrict__ topi, int P, int k, int E,
                                                                   int waves) {
  extern __shared__ int cnt[];           // [waves][E] counts, then cursors
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t run = ((int64_t)P + waves * 64 - 1) / (waves * 64) * 64;
  const int64_t begin = wave < waves ? wave * run : P, end = begin + run < P ? begin + run : P;
  int* mine = cnt + min(wave, waves - 1) * E;
  for (int i = tid; i < waves * E; i += 64 * SORT_WAVES) cnt[i] = 0;
  __syncthreads();
  for (int64_t p0 = begin; p0 < end; p0 += 64) {
    const int64_t p = p0 + lane;
    const int e = p < end ? (int)topi[p] : -1;
    for (int c = 0; c < E; ++c) {
      const unsigned long long m = __ballot(e == c);
      if (m && lane == 0) mine[c] += (int)__popcll(m);
    }
  }
  __syncthreads();
  // an expert's pairs before each run; its whole number in the first run's place
  for (int c = tid; c < E; c += 64 * SORT_WAVES) {
    int at = 0;
    for (int w = 0; w < waves; ++w) {
      const int n = cnt[w * E + c];
      cnt[w * E + c] = at;
      at += n;
    }
    cnt[c] = at;
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
  for (int i = E + tid; i < waves * E; i += 64 * SORT_WAVES) cnt[i] += cnt[i % E];
  __syncthreads();
  for (int64_t p0 = begin; p0 < end; p0 += 64) {
    const int64_t p = p0 + lane;
    const int e = p < end ? (int)topi[p] : -1;
    int place = -1;
    for (int c = 0; c < E; ++c) {
      const unsigned long long m = __ballot(e == c);
      if (!m) continue;
      int first = 0;
      if (lane == 0) first = atomicAdd(&mine[c], (int)__popcll(m));
      first = __shfl(first, 0);
      if (e == c) place = first + (int)__popcll(m & ((1ULL << lane) - 1));
    }
    if (p < end) {
      pos[p] = place;
      if (place >= 0) ids[place] = (int)(p / k);
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

// rows S in sorted space; the grid holds the most tiles that S rows of E experts can make
// on an XCD, eightfold, and a round for shares. Returns 0, or -1 where the LDS cannot be had
template <bool GATEUP>
static int moe_product(void* out, const void* a, const void* w, const int* ids, const void* zeros, const int* offsets,
                       float* part, int* count, int S, int E, int N, int K, hipStream_t stream) {
  if (!tp_lds_ready(reinterpret_cast<const void*>(moe_product_kernel<GATEUP>))) return -1;
  const int64_t n_tiles = GATEUP ? (N + 127) / 128 : (N + 255) / 256;
  const int64_t blocks = (S / 256 + E) * ((n_tiles + 7) / 8) + (part ? TP_SLOTS : 0);
  hipLaunchKernelGGL(moe_product_kernel<GATEUP>, dim3(blocks * 8), dim3(TP_THREADS), TP_LDS, stream, (bf16_t*)out,
                     (const bf16_t*)a, (const bf16_t*)w, ids, (const bf16_t*)zeros, offsets, part, count, E, N, K);
  return 0;
}

extern "C" int launch_moe_gateup(void* act, const void* x, const void* w, const int* sorted_ids, const int* offsets,
                                 const void* zeros, int S, int E, int IN, int K, hipStream_t stream) {
  return moe_product<true>(act, x, w, sorted_ids, zeros, offsets, nullptr, nullptr, S, E, IN, K, stream);
}

extern "C" int launch_moe_down(void* y, const void* act, const void* w, const int* offsets, float* part, int* count,
                               int S, int E, int H, int IN, hipStream_t stream) {
  return moe_product<false>(y, act, w, nullptr, nullptr, offsets, part, count, S, E, H, IN, stream);
}

// Whether the last round's tiles may be shared out: with many rounds it is not worth the room, and of short K their sums'
// way through memory takes longer than it saves. us without and with, the zeros' launch included, 8 experts, top 2, 320 rows:
// width 4096, K 1024 23, 31   2048 46, 51   2560 55, 52   4096 102, 83; width 2048 18, 23   34, 33   54, 40   69, 50. Then floats
// of ``part`` and zeros of ``count``.
extern "C" int64_t moe_down_room(int S, int E, int H, int IN, int* zeros) {
  *zeros = 8 * TP_SLOTS;
  const int64_t tiles = (int64_t)(S / 256 + E) * ((H + 255) / 256);
  return tiles > 8 * 8 * TP_SLOTS || IN < 2560 ? 0 : (int64_t)8 * TP_SLOTS * TP_SUMS;
}

extern "C" void launch_moe_sort(int* ids, int* pos, int* offsets, const int64_t* topi, int P, int k, int E,
                                hipStream_t stream) {
  const int room = 65536 / (int)sizeof(int);       // of LDS
  const int waves = E * SORT_WAVES <= room ? SORT_WAVES : room / E;
  hipLaunchKernelGGL(moe_sort_kernel, dim3(1), dim3(64 * SORT_WAVES), waves * E * sizeof(int), stream, ids, pos, offsets, topi,
                     P, k, E, waves);
}

extern "C" void launch_moe_combine(void* out, const void* y, const float* weights, const int* pos, int T, int k,
                                   int H, hipStream_t stream) {
  const int nvec = H / 8;
  hipLaunchKernelGGL(moe_combine_kernel, dim3(T, (nvec + 255) / 256), dim3(256), 0, stream, (bf16_t*)out,
                     (const bf16_t*)y, weights, pos, k, nvec);
}
