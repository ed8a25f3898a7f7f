// Grouped mixture-of-experts products for gfx950 (prefill shapes):
//
//   moe_route     the router: logits, softmax, the top choices and their weights, in one launch
//   moe_place     the pairs' places grouped by expert, from the counts that moe_route leaves
//   moe_sort      (token, choice) pairs grouped by expert, without the host, for choices made elsewhere
//   moe_gateup    act[s, :] = silu(x[tok(s)] Wg[e]^T) * (x[tok(s)] Wu[e]^T)
//   moe_down      y[s, :]   = act[s] Wd[e]^T
//   moe_combine   out[t, :] = sum over choices j of w[t, j] y[pos(t, j)], in fp32
//
// The products run on the 256-column tiles of tile_product.h: a workgroup computes up to 256
// rows of one expert by 256 columns (gate/up: 128 gate and the same 128 up columns, 64 of each a wave).
//
// What bounds them: with a few hundred rows an expert or fewer, the stream of W from memory;
// above, the matrix units. So the row tiles of an expert are even parts of its rows, in
// tiles of 64, 128, 160, 192, 224 or 256 rows: they keep step, and the 2 or 3 of a column run side
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
// The layer with a router of seven launches at 65 / 150 / 300 / 600 / 1024 / 2048 / 6000 rows, experts of 14336: 582 / 582 /
// 605 / 666 / 949 / 1431 / 3623 us (741 / 760 / 787 / 907 / 1131 / 1935 / 4622); moe_route has what it was after that.
//
// Tiles of 224 rows are for parts of 193 to 224, a tenth less than a tile of 256. The layer, us without them and with: 1600
// rows 1144, 1057; 2600 1720, 1610; experts of 7168, 3300 rows 1105, 1016. When W has the streaming hint: moe_once.

#include "tile_product.h"

// one tile; GATEUP: a = x [T, K] gathered by ids, w [E, 2 * N, K] (gate at [0, N), up behind), out [S, N].
// Down: a = act [S, K], w [E, N, K], out [S, N]
template <bool GATEUP, bool ONCE, int MJ>
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
    const TileRowsOf<ONCE> wr(w + ((int64_t)e * 2 + (wave & 1)) * N * K + k0, n_put, N, 64, K, lane);
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
    const TileRowsOf<ONCE> wr(w + (int64_t)e * N * K + k0, n_put, N, 64, K, lane);
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
template <bool GATEUP, bool ONCE>
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
#define MOE_TILE(MJ) moe_tile<GATEUP, ONCE, MJ>(out, a, w, ids, zeros, e, m0, m_end, n0, N, K, sh, smem)
  if (rows > 224) MOE_TILE(8);
  else if (rows > 192) MOE_TILE(7);
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

// The router of a mixture layer: z = x gate^T rounded to bf16, as the layer's own product gives it, p = softmax(z) in 32
// bits, the k largest (of equal ones the lowest expert, as torch takes them; NaN before all) and their shares of their
// sum. For moe_place: each pair's rank among the group's earlier pairs of its expert, and the group's counts.
//
// A workgroup takes 16 rows, one tile of the matrix cores, and its 16 waves share K, so that a row's loads are all in
// flight at once: with 100 rows the chain of a launch and one trip to memory is the bound, with thousands the stream of
// x. Seven launches of torch's before (product, conversion, softmax, selection of 18 to 24 us, sorting, sum, quotient) and
// moe_sort's single workgroup. us of the layer, before and now, 8 experts, top 2: 80 rows of width 2048 and experts of
// 8192 226, 187; 300 rows 246, 201; 6000 rows 1133, 1061; width 4096 and experts of 7168, 780 rows 426, 385; of 14336,
// 2048 rows 1401, 1348.
#define ROUTE_ROWS 16
#define ROUTE_WAVES 16
#define ROUTE_EXPERTS 32
#define ROUTE_TOP 8

template <int NT>                        // tiles of 16 experts
__global__ void __launch_bounds__(64 * ROUTE_WAVES) moe_route_kernel(
    int* __restrict__ topi, float* __restrict__ topw, int* __restrict__ rank, int* __restrict__ counts,
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ gate, int T, int H, int64_t x_stride, int E, int k) {
  constexpr int DEEP = 4;
  __shared__ float sums[ROUTE_WAVES][ROUTE_ROWS][NT * 16];
  __shared__ int chosen[ROUTE_ROWS * ROUTE_TOP];
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, grp = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int t0 = blockIdx.x * ROUTE_ROWS;
  // 32 contiguous bytes of a row for each lane group, the same order of k in both operands
  const char* xr = (const char*)(x + (int64_t)min(t0 + col, T - 1) * x_stride) + grp * 32;
  const char* gr[NT];
  f32x4 acc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    gr[n] = (const char*)(gate + (int64_t)min(n * 16 + col, E - 1) * H) + grp * 32;
    acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int steps = H / 64;
  for (int s0 = wave; s0 < steps; s0 += ROUTE_WAVES * DEEP) {
    bf16x8_mfma a[DEEP][2], b[DEEP][NT][2];
#pragma unroll
    for (int u = 0; u < DEEP; ++u) {
      const int64_t at = (int64_t)min(s0 + u * ROUTE_WAVES, steps - 1) * 128;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        a[u][h] = *reinterpret_cast<const bf16x8_mfma*>(xr + at + h * 16);
#pragma unroll
        for (int n = 0; n < NT; ++n) b[u][n][h] = *reinterpret_cast<const bf16x8_mfma*>(gr[n] + at + h * 16);
      }
    }
#pragma unroll
    for (int u = 0; u < DEEP; ++u) {
      if (s0 + u * ROUTE_WAVES >= steps) break;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][h], b[u][n][h], acc[n], 0, 0, 0);
    }
  }
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) sums[wave][grp * 4 + r][n * 16 + col] = acc[n][r];
  __syncthreads();
  if (tid < ROUTE_ROWS * 16) {           // 16 lanes a row, experts col, col + 16, ..
    const int row = tid >> 4, t = t0 + row;
    float p[NT], m = -INFINITY, sum = 0.0f;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      float z = 0.0f;
#pragma unroll
      for (int w = 0; w < ROUTE_WAVES; ++w) z += sums[w][row][n * 16 + col];
      p[n] = n * 16 + col < E ? bf16_to_f32(f32_to_bf16(z)) : -INFINITY;
      m = fmaxf(m, p[n]);
    }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      p[n] = n * 16 + col < E ? expf(p[n] - m) : 0.0f;
      sum += p[n];
    }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
    unsigned long long key[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int e = n * 16 + col;
      key[n] = e < E ? (unsigned long long)__float_as_uint(p[n] / sum) << 32 | (uint32_t)~e : 0;
    }
    float total = 0.0f, mine = 0.0f;
    int e_mine = -1;
    for (int j = 0; j < k; ++j) {
      unsigned long long best = key[0];
#pragma unroll
      for (int n = 1; n < NT; ++n) best = key[n] > best ? key[n] : best;
#pragma unroll
      for (int off = 8; off > 0; off >>= 1) {
        const unsigned long long o = __shfl_xor(best, off);
        best = o > best ? o : best;
      }
#pragma unroll
      for (int n = 0; n < NT; ++n)
        if (key[n] == best) key[n] = 0;
      const float q = __uint_as_float((uint32_t)(best >> 32));
      total += q;
      if (j == col) {
        mine = q;
        e_mine = (int)~(uint32_t)best;
      }
    }
    if (col < k) {
      chosen[row * k + col] = t < T ? e_mine : -1;
      if (t < T) {
        topi[(int64_t)t * k + col] = e_mine;
        topw[(int64_t)t * k + col] = mine / total;
      }
    }
  }
  __syncthreads();
  const int pairs = ROUTE_ROWS * k;
  if (tid < pairs && chosen[tid] >= 0) {
    const int e = chosen[tid];
    int n = 0;
    for (int q = 0; q < tid; ++q) n += chosen[q] == e;
    rank[(int64_t)t0 * k + tid] = n;
  } else if (tid >= 512 && tid < 512 + E) {
    int n = 0;
    for (int q = 0; q < pairs; ++q) n += chosen[q] == tid - 512;
    counts[(int64_t)blockIdx.x * E + tid - 512] = n;
  }
}

// moe_route's pairs -> offsets, pos and ids as moe_sort gives them: an expert's pairs in their order. A workgroup adds up
// all groups' counts (6000 rows: 375 groups of 8, read by 256 threads) and places the pairs of 16 groups. ``zeros``: the
// counters of moe_down's shares, cleared on the way
#define PLACE_GROUPS 16
__global__ void __launch_bounds__(256) moe_place_kernel(int* __restrict__ ids, int* __restrict__ pos, int* __restrict__ offsets,
                                                        int* __restrict__ zeros, int n_zeros, const int* __restrict__ topi,
                                                        const int* __restrict__ rank, const int* __restrict__ counts, int T,
                                                        int k, int E) {
  __shared__ int all[ROUTE_EXPERTS], before[ROUTE_EXPERTS], first[PLACE_GROUPS][ROUTE_EXPERTS];
  const int tid = threadIdx.x, e = tid % ROUTE_EXPERTS;
  const int groups = (T + ROUTE_ROWS - 1) / ROUTE_ROWS, g0 = blockIdx.x * PLACE_GROUPS;
  if (blockIdx.x == 0)
    for (int i = tid; i < n_zeros; i += 256) zeros[i] = 0;
  if (tid < ROUTE_EXPERTS) all[tid] = before[tid] = 0;
  __syncthreads();
  if (e < E) {
    int n = 0, n_before = 0;
#pragma unroll 8
    for (int g = tid / ROUTE_EXPERTS; g < groups; g += 256 / ROUTE_EXPERTS) {
      const int c = counts[(int64_t)g * E + e];
      n += c;
      if (g < g0) n_before += c;
    }
    atomicAdd(&all[e], n);
    atomicAdd(&before[e], n_before);
  }
  __syncthreads();
  if (tid < ROUTE_EXPERTS) {
    int upto = all[e];
#pragma unroll
    for (int off = 1; off < ROUTE_EXPERTS; off <<= 1) {
      const int o = __shfl_up(upto, off);
      if (e >= off) upto += o;
    }
    if (blockIdx.x == 0 && e < E) {
      offsets[e + 1] = upto;
      if (e == 0) offsets[0] = 0;
    }
    int at = upto - all[e] + before[e];
#pragma unroll
    for (int i = 0; i < PLACE_GROUPS; ++i) {
      first[i][e] = at;
      if (g0 + i < groups && e < E) at += counts[(int64_t)(g0 + i) * E + e];
    }
  }
  __syncthreads();
  const int64_t p0 = (int64_t)g0 * ROUTE_ROWS * k;
  const int n = (int)min((int64_t)PLACE_GROUPS * ROUTE_ROWS * k, (int64_t)T * k - p0);
  for (int i = tid; i < n; i += 256) {
    const int place = first[i / (ROUTE_ROWS * k)][topi[p0 + i]] + rank[p0 + i];
    pos[p0 + i] = place;
    ids[place] = (int)((p0 + i) / k);
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

// Whether the products load W with the streaming hint, which leaves the caches to x and to act: where the weights of all experts
// are themselves too large for the 256 MB last-level cache, so that no call finds anything of the one before, and few enough
// rows go to an expert that its W is read by one or two row tiles. Smaller ones stay in the cache in part from call to call, and
// the hint gives that up; of many rows act is as large as the cache itself. us plain and with it, 8 experts, width and size of
// an expert:
//   gate/up  1024x4096 (134 MB), 1024 tokens, 2 choices 58, 61   2048x4096 (268 MB) alone 4 tokens 36, 37; 600 56, 58
//            2048x6144 (402 MB) 32 tokens 84, 80; 800 113, 112   2048x8192 (537 MB) 4 tokens 85, 81; 300 117, 107; 800 131, 127
//              but 1024 168, 171; 2048 270, 273      4096x14336 (1879 MB) 32 tokens 341, 316; 800 422, 417
//   down     2048x4096 (134 MB) alone 32 tokens 32, 54; 1024 73, 93   2048x6144 (201 MB) 2048 tokens 141, 157
//            4096x7168 (470 MB) 4 tokens 96, 93; 300 124, 120; 1024 175, 172
//   both     4096x7168 600 tokens 317, 301; 1600 549, 542; 2048 699, 694; 3000 922, 938
//            4096x14336 150 523, 507; 1024 884, 867; 2048 1321, 1309; 3000 1766, 1796; 6000 3212, 3271
#define MOE_ONCE_BYTES ((int64_t)320 << 20)
static bool moe_once(bool gateup, int64_t S, int64_t E, int64_t N, int64_t K) {
  const int64_t bytes = E * (gateup ? 2 : 1) * N * K * 2;
  return bytes >= MOE_ONCE_BYTES && S <= E * (gateup && bytes < 2 * MOE_ONCE_BYTES ? 224 : 512);
}

// rows S in sorted space; the grid holds the most tiles that S rows of E experts can make
// on an XCD, eightfold, and a round for shares. Returns 0, or -1 where the LDS cannot be had
template <bool GATEUP, bool ONCE>
static int moe_product_of(void* out, const void* a, const void* w, const int* ids, const void* zeros, const int* offsets,
                          float* part, int* count, int S, int E, int N, int K, hipStream_t stream) {
  if (!tp_lds_ready(reinterpret_cast<const void*>(moe_product_kernel<GATEUP, ONCE>))) return -1;
  const int64_t n_tiles = GATEUP ? (N + 127) / 128 : (N + 255) / 256;
  const int64_t blocks = (S / 256 + E) * ((n_tiles + 7) / 8) + (part ? TP_SLOTS : 0);
  hipLaunchKernelGGL((moe_product_kernel<GATEUP, ONCE>), dim3(blocks * 8), dim3(TP_THREADS), TP_LDS, stream, (bf16_t*)out,
                     (const bf16_t*)a, (const bf16_t*)w, ids, (const bf16_t*)zeros, offsets, part, count, E, N, K);
  return 0;
}

template <bool GATEUP>
static int moe_product(void* out, const void* a, const void* w, const int* ids, const void* zeros, const int* offsets,
                       float* part, int* count, int S, int E, int N, int K, hipStream_t stream) {
  const auto product = moe_once(GATEUP, S, E, N, K) ? moe_product_of<GATEUP, true> : moe_product_of<GATEUP, false>;
  return product(out, a, w, ids, zeros, offsets, part, count, S, E, N, K, stream);
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

// E up to ROUTE_EXPERTS, k up to ROUTE_TOP and E, H a multiple of 64, rows on 16 bytes; counts: [ceil(T / 16), E]
extern "C" int moe_route_groups(int T) { return (T + ROUTE_ROWS - 1) / ROUTE_ROWS; }

extern "C" void launch_moe_route(int* topi, float* topw, int* rank, int* counts, const void* x, const void* gate, int T, int H,
                                 int64_t x_stride, int E, int k, hipStream_t stream) {
  hipLaunchKernelGGL(E <= 16 ? moe_route_kernel<1> : moe_route_kernel<2>, dim3(moe_route_groups(T)), dim3(64 * ROUTE_WAVES), 0,
                     stream, topi, topw, rank, counts, (const bf16_t*)x, (const bf16_t*)gate, T, H, x_stride, E, k);
}

extern "C" void launch_moe_place(int* ids, int* pos, int* offsets, int* zeros, int n_zeros, const int* topi, const int* rank,
                                 const int* counts, int T, int k, int E, hipStream_t stream) {
  hipLaunchKernelGGL(moe_place_kernel, dim3((moe_route_groups(T) + PLACE_GROUPS - 1) / PLACE_GROUPS), dim3(256), 0, stream, ids,
                     pos, offsets, zeros, n_zeros, topi, rank, counts, T, k, E);
}

extern "C" void launch_moe_combine(void* out, const void* y, const float* weights, const int* pos, int T, int k,
                                   int H, hipStream_t stream) {
  const int nvec = H / 8;
  hipLaunchKernelGGL(moe_combine_kernel, dim3(T, (nvec + 255) / 256), dim3(256), 0, stream, (bf16_t*)out,
                     (const bf16_t*)y, weights, pos, k, nvec);
}
