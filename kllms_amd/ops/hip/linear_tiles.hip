// Products of many rows (prompts) for gfx950, on the 256-column tiles of tile_product.h:
//
//   plain     out [M, N] = x [M, K] w [N, K]^T (+ bias [N])
//   silu      out [M, N] = silu(x wg^T) * (x wu^T), w = [wg; wu] [2 N, K]
//   clamped   out [M, N] = g sigmoid(alpha g) (u + 1), g = min(x wg^T, limit), u = clamp(x wu^T, +-limit)
//
// A workgroup computes 64 to 256 rows by 256 columns (gated: 128 gate and the same 128 up columns, 64 of each a wave);
// the activation works on the fp32 sums, without gate and up in memory.
//
// What bounds them: the matrix units, at what the power limit leaves of them, and whole rounds of the chip's 256
// compute units. A tile of 32 * MJ rows takes LT_COST[MJ] us for 64 stages of K, so the rows of a tile are those
// whose rounds cost least (4096 rows of N = K = 4096: 256 tiles of 256; 3100 rows: 224 of 224, 77 us, 88 with 256).
// Of long K the tiles of a last round that would leave half of the units idle are shared out over it. The library has
// the advantage where its tiles fill the last round too, and at middling K on few tiles, which it splits and makes
// smaller; linear_tiles_rows has the lines. Measured, us of the library (with its activation's launch) and here:
//   N 4096, K 14336       1170 rows 146, 130    1600 rows 330, 168     3100 rows 334, 280    11700 rows 1303, 1019
//   N 4096, K 4096        3100 rows  82,  77    4700 rows 139, 125    11700 rows  442,  276
//   silu N 14336, K 4096   300 rows  81,  72     777 rows 189, 167    3100 rows 698, 557    11700 rows 2099, 2011
//   silu N 8192, K 2048    300 rows  36,  32     777 rows  61,  51    4700 rows 347, 253     7777 rows  454,  403
//   N 8720, K 2048        1200 rows  48,  43    3300 rows 138, 107     7777 rows 240, 220

#include "tile_product.h"

#define LT_BAND 8          // row tiles of a band: 8 x 4 tiles are in work on an XCD at a time

enum { LT_PLAIN = 0, LT_SILU = 1, LT_CLAMPED = 2 };

// exp(x) to fp32's last places: the rounding of x * log2(e), with that constant split into a high and a low part, is made
// good where it counts: not above fp32's range, nor below it, where an infinite product would leave nothing of the rest
__device__ __forceinline__ float lt_exp(float x) {
  const float t = x * 1.44269504088896341f;
  const float rest = __builtin_fmaf(x, 1.44269504088896341f, -t) + x * 1.92596299112661746e-8f;
  const float e = __builtin_amdgcn_exp2f(t);
  return fabsf(t) < 126.0f ? __builtin_fmaf(e, rest * 0.693147180559945309f, e) : e;
}

template <int ACT, int MJ>
__global__ void __launch_bounds__(TP_THREADS, 1) linear_tiles_kernel(bf16_t* __restrict__ out, const bf16_t* __restrict__ x,
                                                                     const bf16_t* __restrict__ w,
                                                                     const bf16_t* __restrict__ bias, float* __restrict__ part,
                                                                     int* __restrict__ count, int M, int N, int K,
                                                                     int m_tiles, float limit, float alpha) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  constexpr int BN = ACT ? 128 : 256;              // output columns of a workgroup
  const int n_tiles = (N + BN - 1) / BN;
  // an XCD's tiles are neighbours, in bands of rows and column by column in them: those in work at a time share
  // rows of x and of w in its L2
  const int xcd = blockIdx.x & 7;
  const int all = m_tiles * n_tiles;
  const int begin = (int)((int64_t)all * xcd / 8), tiles = (int)((int64_t)all * (xcd + 1) / 8) - begin;
  const TileShare sh(blockIdx.x >> 3, tiles, K / TP_K, part, count, xcd, 256 * 32 * MJ);
  if (sh.tile >= tiles) return;
  const int tile = begin + sh.tile;
  const int bands = (m_tiles + LT_BAND - 1) / LT_BAND, deep = (m_tiles + bands - 1) / bands;
  const int band = tile / (deep * n_tiles), in = tile % (deep * n_tiles);
  const int high = min(deep, m_tiles - band * deep);
  const int rows = (M + m_tiles - 1) / m_tiles;    // even parts
  const int m0 = (band * deep + in % high) * rows, m_end = min(M, m0 + rows);
  const int n0 = in / high * BN;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  f32x4 acc[8][MJ];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int stages = sh.length(K / TP_K);
  const int64_t k0 = (int64_t)sh.first(K / TP_K) * TP_K;
  const int m = m0 + (wave & 1) * MJ * 16;         // first row of this wave's results
  const int m_put = m0 + wave * MJ * 8;
  const TileRows xr(x + k0, m_put, m_end, MJ * 8, K, lane);
  // W rows of a gated tile: 64 gate, 64 up, the next 64 gate, 64 up
  const int n_put = ACT ? n0 + (wave >> 1) * 64 : n0 + wave * 64;
  const TileRows wr(w + (ACT ? (int64_t)(wave & 1) * N : 0) * K + k0, n_put, N, 64, K, lane);
  // the XCDs begin at different k: rows of a power of two of bytes would have all of them at the same memory channels
  tile_product<MJ>(acc, wr, xr, stages, stages * xcd / 8, smem);
  if (sh.shares > 1 && !tile_fold<MJ>(acc, sh.part, sh.share, sh.shares, sh.count, smem)) return;
  if constexpr (ACT != LT_PLAIN) {
    const int n = n0 + (wave >> 1) * 64;
    tile_store<4, MJ>(out + (int64_t)m * N + n, N, m_end - m, N - n, smem, [&](int i, int j) {
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float g = acc[i][j][r], u = acc[i + 4][j][r];
        if constexpr (ACT == LT_SILU) {
          v[r] = g / (1.0f + __expf(-g)) * u;
        } else {
          g = fminf(g, limit);
          u = fminf(fmaxf(u, -limit), limit);
          v[r] = g / (1.0f + lt_exp(-alpha * g)) * (u + 1.0f);
        }
      }
      return tp_pack(v[0], v[1], v[2], v[3]);
    });
  } else {
    const int n = n0 + (wave >> 1) * 128;
    const int grp = lane >> 4;
    tile_store<8, MJ>(out + (int64_t)m * N + n, N, m_end - m, N - n, smem, [&](int i, int j) {
      bf16x4_vec b = {0, 0, 0, 0};
      if (bias && n + i * 16 + grp * 4 < N)        // whole units of 4: N is a multiple of 8
        b = *reinterpret_cast<const bf16x4_vec*>(bias + n + i * 16 + grp * 4);
      return tp_pack(acc[i][j][0] + bf16_to_f32(b[0]), acc[i][j][1] + bf16_to_f32(b[1]), acc[i][j][2] + bf16_to_f32(b[2]),
                     acc[i][j][3] + bf16_to_f32(b[3]));
    });
  }
}

template <int ACT, int MJ>
static int linear_tiles_launch(void* out, const void* x, const void* w, const void* bias, float* part, int* count, int M,
                               int N, int K, float limit, float alpha, hipStream_t stream) {
  if (!tp_lds_ready(reinterpret_cast<const void*>(linear_tiles_kernel<ACT, MJ>))) return -1;
  constexpr int BN = ACT ? 128 : 256;
  const int m_tiles = (M + 32 * MJ - 1) / (32 * MJ);
  const int64_t all = (int64_t)m_tiles * ((N + BN - 1) / BN);
  hipLaunchKernelGGL((linear_tiles_kernel<ACT, MJ>), dim3(((all + 7) / 8 + (part ? TP_SLOTS : 0)) * 8), dim3(TP_THREADS), TP_LDS,
                     stream, (bf16_t*)out, (const bf16_t*)x, (const bf16_t*)w, (const bf16_t*)bias, part, count, M, N, K, m_tiles, limit, alpha);
  return 0;
}

// us of a round of tiles of 32 * MJ rows by 256 columns and 64 stages of K, with all compute units at work
static const int LT_COST[9] = {0, 0, 44, 49, 60, 68, 77, 88, 97};
#define LT_UNITS (8 * TP_SLOTS)
#define LT_LONG 8192       // K from which the last round's tiles may be shared out

// MJ of the tiles of a product, + 16 where the last round is shared out over K, or 0 where the library's is the better
// one; N: columns of the result
extern "C" int linear_tiles_rows(int64_t M, int64_t N, int64_t K, int act) {
  const int64_t n_tiles = act ? (N + 127) / 128 : (N + 255) / 256, stages = K / TP_K;
  int best = 8;
  double least = 1e30;
  for (int mj = 8; mj >= 2; --mj) {
    const int64_t tiles = (M + 32 * mj - 1) / (32 * mj) * n_tiles;
    const double round = LT_COST[mj] * (K / 4096.0);
    const double whole = (tiles + LT_UNITS - 1) / LT_UNITS * round;
    if (whole < least) least = whole, best = mj;
    const int64_t unit = (tiles + 7) / 8, rest = unit % TP_SLOTS;
    if (K < LT_LONG || rest == 0 || rest > TP_SLOTS / 2) continue;
    const int64_t shares = TP_SLOTS / rest < TP_SHARES ? TP_SLOTS / rest : TP_SHARES;
    // the sums' way through memory: 16 us for four shares of 64 rows, 28 for three of 256
    const double shared = unit / TP_SLOTS * round + round / (shares < stages / 8 ? shares : stages / 8) + 10 + 0.75 * mj * shares;
    if (shared < least) least = shared, best = mj + 16;
  }
  // few rows: the weights' stream bounds, which one tile a column does not keep up
  if (M <= 128) return 0;
  // Few tiles: the library splits K and makes its tiles smaller. Where both are even (us of the library and here, in a
  // graph), by results: at K 2048 from 3.5 million (N 2048: 11 and 19 at 300 rows, 20.0 and 20.3 at 1200, 29.8 and 24.5 at
  // 2600; N 8720: 25 and 28 at 300, 30.7 and 30.6 at 465, 48 and 43 at 1200), at K 4096 from 6.5 (N 4096: 26 and 54 at 300, 48 and 53
  // at 1200, 58.5 and 56.8 at 1600). Longer K is shared out (N 4096, K 14336: 63 and 63 at 256 rows, 78 and 67 at
  // 300, 325 and 176 at 1600; N 2048, K 8192: 34 and 36 at 400, 44 and 42 at 600). Gated products save the activation's
  // launch and pass: ahead from the start at K 2048 (16384 rows of w: 31 and 29 at 140), later at K 4096 (28672: 67 and 69
  // at 140, 80 and 71 at 200)
  const int64_t outputs = M * N * (act ? 2 : 1);
  const int64_t least_outputs = K >= LT_LONG ? 1200000 : act ? (K > 2048 ? 5000000 : 0) : K > 2048 ? 6500000 : 3500000;
  if (outputs < least_outputs) return 0;
  // 256 x 256 tiles that fill one or two rounds to 0.92 and more: the library's are 4 to 10 % faster (N 4096, K 4096 /
  // 14336: 3710 rows 94 and 99 / 309 and 339, 8100 rows 184 and 200 / 619 and 699). Below it is not, on balance (2700
  // rows 78 and 77 / 249 and 253; 4200 rows 140 and 125 / 730 and 377; 7600 rows 179 and 195 / 1009 and 696), and
  // of three rounds and more, or where a tile is short, it is seldom (12000 rows 450 and 297 / 1359 and 1067)
  const int64_t tiles = (M + 255) / 256 * n_tiles;
  const int64_t last = tiles % LT_UNITS ? tiles % LT_UNITS : LT_UNITS;
  if (!act && K > 2048 && tiles <= 2 * LT_UNITS && last * 25 >= LT_UNITS * 23) return 0;
  return best;
}

// floats of part and zeros of count that shares take
extern "C" int64_t linear_tiles_room(int mj, int* zeros) {
  *zeros = LT_UNITS;
  return (int64_t)LT_UNITS * 256 * 32 * mj;
}

// 0, or -1 where the LDS cannot be had
extern "C" int launch_linear_tiles(void* out, const void* x, const void* w, const void* bias, float* part, int* count, int M,
                                   int N, int K, int act, int mj, float limit, float alpha, hipStream_t stream) {
#define LT_CASE(MJ)                                                                                           \
  case MJ:                                                                                                    \
    return act == LT_SILU      ? linear_tiles_launch<LT_SILU, MJ>(out, x, w, bias, part, count, M, N, K, limit, alpha, stream)    \
           : act == LT_CLAMPED ? linear_tiles_launch<LT_CLAMPED, MJ>(out, x, w, bias, part, count, M, N, K, limit, alpha, stream) \
                               : linear_tiles_launch<LT_PLAIN, MJ>(out, x, w, bias, part, count, M, N, K, limit, alpha, stream)
  switch (mj) {
    LT_CASE(2);
    LT_CASE(3);
    LT_CASE(4);
    LT_CASE(5);
    LT_CASE(6);
    LT_CASE(7);
    LT_CASE(8);
    default:
      return -1;
  }
#undef LT_CASE
}
