// Products of a few rows with a weight matrix, y[M, N] = x[M, K] W[N, K]^T (the projections of a decode step or of a
// short prompt), for gfx950, on the ring of tile_product.h.
//
// The weights' stream is the bound, and bytes in flight are what keeps it up: W and x go from memory to LDS without
// registers in between, 64 deep in k, and a workgroup has all its buffers on their way from its first instruction on -
// 60 to 150 KB of a compute unit. (Weights loaded to registers two to four chunks ahead, with x through two LDS buffers,
// streamed 28672 x 4096 at 4.6 TB/s for 5 rows and at 3.4 for 96; so it is 5.7 and 5.2, 6.2 with the streaming hint.) A workgroup takes 64 or 128 rows of
// W; MJ tiles of 32 rows of x are multiplied at once, so that LDS is read once for 16 * MJ rows and not for 16.
//
// A matrix of few rows is also split over k (linear_rows_splits); the splits' fp32 sums are left to the consumer, which
// reads them anyway (rope + store, residual + norm). Forms of the result:
//   PART  fp32 sums [S, M, N]          SILU  silu(gate) * up of a fused [gate; up] matrix
//   F32   fp32, S = 1 (logits)         CLAMPED  the clamped gated form of the hybrid family
//   BF16  rounded once, bias added before it
//
// Measured in graphs, weights out of cache, us with the weights through registers and so, both without the streaming hint of
// large matrices (LR_ONCE has what that gives):
//   PART  4096 x 4096   5 rows 8.5, 8.1   40 rows 10.0, 8.7   96 14.3, 11.0     6144 x 4096   5 rows 11.6, 11.1   64 15.9, 12.9
//     4096 x 14336   5 rows 23.7, 23.3   40 26.4, 24.9   96 35.0, 30.6     2048 x 8192   16 rows 9.2, 8.6   128 16.6, 12.4
//     2048 x 2048   5 rows 3.9, 4.3   128 7.4, 6.2
//   SILU  28672 x 4096   5 rows 51.0, 41.0   64 55.7, 42.7   128 69.2, 50.0 (library and activation 60.2)
//     16384 x 2048   1 row 17.6, 13.5   40 20.1, 13.7   96 29.2, 16.4 (22.3)
//   F32   32000 x 4096   5 rows 54.6, 44.8 (library 59.9)   128 76.8, 59.8 (65.4)     128256 x 4096   1 row 202.7, 176.9 (188.7)
// and against the library above 128 rows:
//   PART  4096 x 4096   192 rows 32.8, 14.6   256 23.3, 17.5   384 25.2, 22.6     4096 x 14336   192 103, 39.4   384 82.4, 55.6
//   SILU  28672 x 4096   160 rows 63.4, 53.5   256 72.6, 63.5     16384 x 2048   192 31.1, 22.3   256 35.3, 25.8

#include <atomic>

#include "tile_product.h"

enum LinearForm { LR_PART = 0, LR_BF16 = 1, LR_F32 = 2, LR_SILU = 3, LR_CLAMPED = 4 };

// Workgroups by share of k, then by rows of W, then by rows of x: those of an XCD have the same part of x in its L2, and
// the row tiles of a part of W run side by side.
// more: the bias (BF16), or a second matrix (PART): then K is both matrices' and the halves of the splits are two products, of
// x's first M rows with w and of the next M with more. ONCE: W passes the caches by (LR_ONCE)
template <int NI, int MJ, int FORM, int KB, bool ONCE>
__global__ void __launch_bounds__(TP_THREADS, 1) linear_rows_kernel(
    void* __restrict__ out, const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, const bf16_t* __restrict__ more,
    int M, int N, int K, int x_stride, int m_tiles, int splits, float limit, float alpha) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  constexpr bool GATED = FORM == LR_SILU || FORM == LR_CLAMPED;
  constexpr int BN = GATED ? 16 * NI : 32 * NI;    // columns of the result
  const int columns = GATED ? N / 2 : N;
  const int n_tiles = (columns + BN - 1) / BN, all = n_tiles * splits * m_tiles, xcd = blockIdx.x & 7;
  const int begin = (int)((int64_t)all * xcd >> 3), items = (int)((int64_t)all * (xcd + 1) >> 3) - begin;
  const int at = blockIdx.x >> 3;
  if (at >= items) return;
  const int item = begin + at, rest = item / m_tiles, share = rest / n_tiles, n0 = rest % n_tiles * BN;
  const int rows = (M + m_tiles - 1) / m_tiles;    // even parts
  const int m0 = item % m_tiles * rows, m_end = min(M, m0 + rows);
  const uint32_t stages_all = K / TP_K, first = stages_all * share / splits;      // both far below 2^16
  const int stages = (int)(stages_all * (share + 1) / splits - first);
  const int64_t k0 = (int64_t)first * TP_K;
  const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  f32x4 acc[NI][MJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // W rows of a gated tile: 8 * NI gate, the same of up, the next gate, their up
  const int n_put = GATED ? n0 + (wave >> 1) * (8 * NI) : n0 + wave * (8 * NI);
  const bf16_t* wk = w + (GATED ? (int64_t)(wave & 1) * columns : 0) * K + k0;
  const bf16_t* xk = x + k0;
  int w_row = K;
  if constexpr (FORM == LR_PART) {
    if (more) {
      w_row = K / 2;
      if (2 * share >= splits) {
        wk = more + (k0 - w_row);
        xk += (int64_t)M * x_stride - w_row;
      }
    }
  }
  const TileRows xr(xk, m0 + wave * MJ * 8, m_end, MJ * 8, x_stride, stages * TP_K, lane);
  const TileRowsOf<ONCE> wr(wk, n_put, columns, 8 * NI, w_row, lane);
  // the XCDs begin at different k: rows of a power of two of bytes would have all of them at the same memory channels
  tile_product<MJ, NI, KB * 1024>(acc, wr, xr, stages, stages * xcd / 8, smem);
  if constexpr (FORM == LR_SILU && MJ > 4) {       // many rows: whole lines
    const int m = m0 + (wave & 1) * MJ * 16, n = n0 + (wave >> 1) * (BN / 2);
    tile_store<NI / 2, MJ>((bf16_t*)out + (int64_t)m * columns + n, columns, m_end - m, columns - n, smem, [&](int i, int j) {
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float g = acc[i][j][r];
        v[r] = g / (1.0f + __expf(-g)) * acc[i + NI / 2][j][r];
      }
      return tp_pack(v[0], v[1], v[2], v[3]);
    });
    return;
  }
  const int m = m0 + (wave & 1) * MJ * 16 + col, n = n0 + (wave >> 1) * (BN / 2) + grp * 4;
#pragma unroll
  for (int j = 0; j < MJ; ++j) {
    const int mr = m + j * 16;
    if (mr >= m_end) continue;
#pragma unroll
    for (int i = 0; i < (GATED ? NI / 2 : NI); ++i) {
      const int nc = n + i * 16;
      if (nc >= columns) continue;
      if constexpr (GATED) {
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float g = acc[i][j][r], u = acc[i + NI / 2][j][r];
          if constexpr (FORM == LR_SILU) {
            v[r] = g / (1.0f + __expf(-g)) * u;
          } else {
            const float gc = fminf(g, limit), uc = fminf(fmaxf(u, -limit), limit);
            v[r] = gc * (1.0f / (1.0f + expf(-alpha * gc))) * (uc + 1.0f);
          }
        }
        *reinterpret_cast<bf16x4_vec*>((short*)out + (int64_t)mr * columns + nc) = tp_pack(v[0], v[1], v[2], v[3]);
      } else if constexpr (FORM == LR_BF16) {
        bf16x4_vec o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = f32_to_bf16(acc[i][j][r] + (more ? bf16_to_f32(((const short*)more)[nc + r]) : 0.0f));
        *reinterpret_cast<bf16x4_vec*>((short*)out + (int64_t)mr * N + nc) = o;
      } else {
        *reinterpret_cast<f32x4*>((float*)out + ((int64_t)share * M + mr) * N + nc) = acc[i][j];
      }
    }
  }
}

#define LR_UNITS 256       // compute units

// Tiles of a product: rows of W 32 * ni, rows of x 32 * mj in m_tiles parts, KB of LDS (80: two workgroups to a compute
// unit, whose streams fill each other's beginnings and ends).
struct LinearPlan {
  int ni, mj, m_tiles, kb;
};

// Up to 128 rows one part of x, so that W is read once; above, two or more read it from the L2 where the splits they
// replace would cost more in sums (4096 x 4096, 384 rows, with the sums' reading: four parts in two splits 25.1 us, one in
// eight above 30). Four parts of a small matrix, three of a wider one, two from N 4096 or 2^24 weights on: these leave it fewer
// splits in any case, and each part reads all of W. us with the sums' reading, in parts of up to 96 rows and so, library last, at
// 160 / 256 / 320 / 384 rows:
//   2048 x 2048  15.4 12.3 15 / 16.2 14.3 15 / 17.7 17.4 17 / 19.0 18.7 16    1024 x 4096  16.0 12.4 15 / 21.3 14.6 15 / 17.7 17.5 18 / 19.2 19.1 19
//   3072 x 3072  18.3 17.0 20 / 20.5 20.5 22 / 24.8 22.9 22 / 25.9 26.1 24    3072 x 8192  26.0 25.7 32 / 31.2 28.7 38 / 40.4 32.8 38 / 42.8 35.2 47
//   3072 x 12288  37.1 36.7 48 / 45.4 42.6 56 / 67.5 46.8 57 / 71.3 50.0 73   3584 x 18944  54.1 53.6 111 / 63.9 62.7 130 / 83.2 66.7 86 / 88.2 72.3 89
// 64 rows of W to a tile where 128 would leave half of the compute units idle (4096 x 4096, 5 rows: 8.0 us, 8.4; silu
// 16384 x 2048 13.5, 15.2; but 18432 x 4096, 144 tiles of 128 rows, 35.2, 30.7) or make more workgroups than there are (silu
// 37888 x 3584, 16 rows: 57, 64), and of PART up to N 5632, and near 8192 at few rows, where they fill the compute units as well
// (with 128 rows and with 64: 5120 x 5120 1 row 17.1, 15.4   128 28.5, 26.8; 8192 x 6144 1 row 28.0, 26.8; but 6144 x 6144 128 rows
// 31.1, 38.7); 128 of a long matrix at many rows of x, whose reading by all of them weighs more (4096 x 14336, 128 rows: 40.8 us
// with the sums' reading, 37.9; 5120 x 13824, 96 rows 40.3, 38.7).
static LinearPlan linear_plan(int M, int N, int K, int form) {
  LinearPlan p;
  const bool gated = form == LR_SILU || form == LR_CLAMPED;
  if (M <= 128) {
    p.m_tiles = 1;
    p.mj = (M + 31) / 32;
    if (form == LR_PART)
      p.ni = (N <= 5632 && !(p.mj == 4 && N >= 4096 && K >= 8192) && !(N >= 5120 && K > 8192)) ||
                     (p.mj == 1 && N >= 7680 && N <= 8448) ? 2 : 4;
    else if (gated)
      p.ni = N <= 256 * 64 || (N > 256 * 128 && p.mj == 1) ? 2 : 4;
    else
      p.ni = p.mj > 1 && N >= 192 * 128 ? 4 : 2;
  } else {
    p.ni = 4;
    p.m_tiles = gated ? (N > 256 * 64 ? 1 : 2) : N >= 4096 || (int64_t)N * K >= 1 << 24 ? 2 : N >= 3072 ? 3 : 4;
    p.mj = ((M + p.m_tiles - 1) / p.m_tiles + 31) / 32;
  }
  p.kb = p.ni == 2 || p.mj <= 2 ? 80 : 160;
  return p;
}

// room for the kernel's LDS; the attribute is asked for once a device
static bool lr_lds_ready(const void* kernel, std::atomic<uint64_t>& devices) {
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return false;
  const uint64_t bit = 1ull << (device & 63);
  if (device < 64 && (devices.load(std::memory_order_relaxed) & bit)) return true;
  if (!tp_lds_ready(kernel)) return false;
  if (device < 64) devices.fetch_or(bit, std::memory_order_relaxed);
  return true;
}

// Whether W's rows are loaded with the streaming hint (nt): where the caller says that the weights of its step are too large to
// stay in the last-level cache (256 MB) until the next one, or the matrix is by itself. Without the hint such weights push out of
// it, and of the L2, what the step reads again (x, sums, keys of shared prompts) and hit nothing themselves. us without and with:
//   SILU  16384 x 2048   1 row 14.3, 12.8 with 335 MB of weights in turn   13.8, 12.5 with 870   128 rows 19.1, 18.6   18.6, 18.2
//   PART  2048 x 8192   1 row 8.5, 8.1 with 301 MB   8.4, 7.8 with 870   128 rows 12.7, 12.8   12.5, 12.3
//     4096 x 4096   1 row 8.1, 7.9   8.0, 7.6   128 rows 13.2, 13.2   13.0, 12.8     4096 x 14336   5 rows 23.8, 20.9 with 900 MB
//   SILU  28672 x 4096   5 rows 41.6, 37.6 (6.2 TB/s)   120 49.6, 46.9   256 64.3, 63.5 with 900 MB     F32   32000 x 4096   5 rows
//     46.6, 41.3   120 54.9, 51.7
// Weights that do fit lose by it: with 200 MB 16384 x 2048 1 row 12.5, 12.3   128 rows 14.3, 18.9; 2048 x 8192 8.0, 8.5   10.3, 12.9;
// 8192 x 1024 6.0, 6.9   8.1, 10.7; between 268 and 290 MB it depends on the rows. Matrices of less than LR_ONCE are plain
// always: nobody waits for them.
#define LR_ONCE (8 << 20)
#define LR_ONCE_ALONE ((int64_t)320 << 20)

template <int NI, int MJ, int FORM, int KB, bool ONCE>
static int linear_rows_go(void* out, const bf16_t* x, const bf16_t* w, const bf16_t* more, int M, int N, int K, int x_stride,
                          int m_tiles, int splits, float limit, float alpha, hipStream_t stream) {
  static std::atomic<uint64_t> devices{0};
  if (!lr_lds_ready(reinterpret_cast<const void*>(linear_rows_kernel<NI, MJ, FORM, KB, ONCE>), devices)) return -1;
  constexpr int LDS = TileRing<MJ, NI, KB * 1024>::STRIDE * TileRing<MJ, NI, KB * 1024>::RING;
  const int64_t all = (int64_t)((N + 32 * NI - 1) / (32 * NI)) * splits * m_tiles;
  hipLaunchKernelGGL((linear_rows_kernel<NI, MJ, FORM, KB, ONCE>), dim3((all + 7) / 8 * 8), dim3(TP_THREADS), LDS, stream, out, x, w, more,
                     M, N, K, x_stride, m_tiles, splits, limit, alpha);
  return 0;
}

template <int FORM>
static int linear_rows_form(const LinearPlan& p, void* out, const bf16_t* x, const bf16_t* w, const bf16_t* more, int M, int N,
                            int K, int x_stride, int splits, float limit, float alpha, bool once, hipStream_t stream) {
  const int64_t bytes = (int64_t)N * K * (int64_t)sizeof(bf16_t);     // of two matrices K is both's
  once = once ? bytes >= LR_ONCE : bytes >= LR_ONCE_ALONE;
#define LR_CASE(NI, MJ)                                                                                              \
  if (p.ni == NI && p.mj == MJ)                                                                                      \
    return once ? linear_rows_go<NI, MJ, FORM, (NI == 2 || MJ <= 2 ? 80 : 160), true>(out, x, w, more, M, N, K, x_stride, p.m_tiles, \
                                                                                      splits, limit, alpha, stream)  \
                : linear_rows_go<NI, MJ, FORM, (NI == 2 || MJ <= 2 ? 80 : 160), false>(out, x, w, more, M, N, K, x_stride, p.m_tiles, \
                                                                                       splits, limit, alpha, stream)
  LR_CASE(2, 1);
  LR_CASE(2, 2);
  LR_CASE(2, 3);
  LR_CASE(2, 4);
  LR_CASE(4, 1);
  LR_CASE(4, 2);
  LR_CASE(4, 3);
  LR_CASE(4, 4);
  if constexpr (FORM == LR_PART || FORM == LR_SILU) {
    LR_CASE(4, 5);
    LR_CASE(4, 6);
  }
  if constexpr (FORM == LR_SILU) {
    LR_CASE(4, 7);
    LR_CASE(4, 8);
  }
#undef LR_CASE
  return -1;
}

// Rows up to which a form is taken
extern "C" int linear_rows_most(int form) { return form == LR_PART ? 384 : form == LR_SILU ? 256 : 128; }

// x_stride from which on 64 rows' offsets would leave 32 bits
extern "C" int64_t linear_rows_strides() { return 1 << 25; }

// 0, or -1 where the LDS cannot be had. x_stride: any below linear_rows_strides(), 0 and less than K too; once: the weights of
// the caller's step pass the caches by (LR_ONCE)
extern "C" int launch_linear_rows(void* out, const bf16_t* x, const bf16_t* w, const bf16_t* bias, int M, int N, int K,
                                  int x_stride, int form, int splits, float limit, float alpha, bool once, hipStream_t stream) {
  const LinearPlan p = linear_plan(M, N, K, form);
#define LR_FORM(F) \
  case F: return linear_rows_form<F>(p, out, x, w, bias, M, N, K, x_stride, splits, limit, alpha, once, stream)
  switch (form) {
    LR_FORM(LR_PART);
    LR_FORM(LR_BF16);
    LR_FORM(LR_F32);
    LR_FORM(LR_SILU);
    LR_FORM(LR_CLAMPED);
  }
#undef LR_FORM
  return -1;
}

// splits of k for the PART form: one workgroup for each compute unit, and four stages of 64 at least
extern "C" int linear_rows_splits(int M, int N, int K) {
  const LinearPlan p = linear_plan(M, N, K, LR_PART);
  const int tiles = (N + 32 * p.ni - 1) / (32 * p.ni) * p.m_tiles, most = K / TP_K / 4;
  const int s = (LR_UNITS + 8) / tiles;
  return s < 1 || most < 1 ? 1 : s < most ? s : most;
}

// PART sums of two products of one size, x [2, M, K] with w and w2 [N, K]: [S, M, N], the first half of the (even) S the one's
extern "C" int launch_linear_rows_two(float* out, const bf16_t* x, const bf16_t* w, const bf16_t* w2, int M, int N, int K,
                                      int splits, bool once, hipStream_t stream) {
  return linear_rows_form<LR_PART>(linear_plan(M, N, K, LR_PART), out, x, w, w2, M, N, 2 * K, K, splits, 0.0f, 0.0f, once, stream);
}
