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
// the advantage where its tiles fill the last round too, and on few tiles, which it splits over K and makes
// smaller; linear_tiles_ahead has the lines. Measured, us of the library (with its activation's launch) and here:
//   N 4096, K 14336       1170 rows 146, 130    1600 rows 330, 168     3100 rows 334, 280    11700 rows 1303, 1019
//   N 4096, K 4096        4700 rows 139, 125    11700 rows  442,  276
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

// Whether the product is faster here than in the library; rows: of w. The library's time goes by tiles of 256 x 256 in
// rounds of the compute units as well: by how many rounds they make, and how much of them they fill. Few tiles it splits
// over K and makes smaller; its third and fifth round cost as much as the next one, and from K 10240 on its short rounds
// do; where w's rows are no multiple of 256, all do. Gated products save the activation's launch and pass here.
//
// Measured in graphs at 78000 sizes, K 64 to 28672, N 256 to 18944, 129 to 12000 rows, us of the library and here:
//   plain, one round     K 4096, N 4096: 1196 rows 49, 51   2021 66, 64   3493 95, 97     K 2048, N 8192: 593 rows 28, 31
//     1969 52, 66       K 2048, N 3072: 1755 rows 27, 25    K 14336, N 4096: 521 rows 112, 82    2455 233, 235    3974 304, 345
//   plain, two           K 2048, N 3072: 5922 rows 83, 70   8984 95, 98    K 4096, N 14336: 1545 rows 159, 167
//   plain, three, four   K 4096, N 4096: 9513 rows 345, 251    11949 448, 286    N 14336: 3179 rows 431, 298    3702 434, 354
//   plain, ragged        N 3216, K 2048: 1206 rows 27, 23   4021 59, 46    7710 134, 89
//   gated                K 1024, N 512: 306 rows 11, 12   2513 17, 13    K 2048, N 1024: 357 rows 14, 19   1124 23, 20
//     K 4096, N 2048: 339 rows 27, 47   1203 55, 50    K 7168, N 4096: 711 rows 92, 100   3207 315, 313
// Of the sizes, 35 % of the plain and 71 % of the gated products are taken: 1.18 and 1.27 times as fast in the mean, 13
// and 4 % of them slower by 3 % or more. (With a least number of results alone, stepped at K 2048, 4096 and 8192, 55 and
// 84 % were: 1.11 and 1.21, 25 and 11 % slower.)
static bool linear_tiles_ahead(int64_t M, int64_t rows, int64_t K, bool gated) {
  // the weights' stream bounds few rows, and one tile a column does not keep it up
  if (M <= 128) return false;
  const int64_t tiles = (M + 255) / 256 * ((rows + 255) / 256), rounds = (tiles + LT_UNITS - 1) / LT_UNITS;
  const double fill = (double)tiles / (rounds * LT_UNITS);
  const bool ragged = rows % 256 != 0;
  if (K >= 10240) {                                // the last round shared out over K here
    if (rounds == 1)
      return fill > (M >= 700 || K >= 16384 ? 0.08 : 0.1) && fill <= (M >= 700 || gated || K >= 16384 ? 0.5 : 0.25);
    if (rounds == 2 || (rounds == 4 && !gated)) return fill <= 0.92;
    return gated || rounds <= 5;
  }
  if (gated) {
    if (K <= 1280) return rounds > 1 || fill > 0.05;
    if (K <= 2304) return rounds > 1 || fill > 0.2;
    if (rounds == 1) return K <= 4608 ? fill > (M >= 700 ? 0.3 : 0.4) : M >= 1500 && fill > 0.3 && fill <= 0.84;
    return rounds > 2 || ragged || fill <= (K <= 4608 ? 0.84 : 0.92);
  }
  if (ragged && K >= 256) {
    if (rounds == 1) return K <= 1280 ? fill > 0.25 : K <= 4608 ? fill > 0.5 : K < 8192 && fill > 0.7 && fill <= 0.84;
    return K <= 4608 || rounds <= (K < 8192 ? 5 : 4);
  }
  if (K <= 640) return K >= 256 && (rounds > 1 || fill > 0.25) && fill <= 0.92;
  if (rounds == 1) return M >= (K < 8192 ? 1500 : 4000) && fill >= (K <= 2048 ? 0.25 : K < 8192 ? 0.4 : 0.5) && fill <= 0.7;
  if (rounds == 2) return fill <= 0.7;
  if (rounds == 4) return fill <= 0.84;
  return (rounds == 3 || rounds == 5) && fill <= (K >= 2048 ? 0.99 : 0.84);
}

// MJ of the tiles of a product, + 16 where the last round is shared out over K, or 0 where the library's is the better
// one; N: columns of the result
extern "C" int linear_tiles_rows(int64_t M, int64_t N, int64_t K, int act) {
  if (!linear_tiles_ahead(M, act ? 2 * N : N, K, act != 0)) return 0;
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
