// Products of a few rows with a weight matrix, y[M, N] = x[M, K] W[N, K]^T, M <= 128
// (the projections of a decode step), for gfx950.
//
// The weights' stream is the bound: 64 weight rows per 256-thread workgroup (128 per 512
// for many rows of x), 16 per wave, each read once and straight from memory to matrix fragments (16x16x32) - a
// lane group takes 32 contiguous bytes of its row in two loads, so every 128-byte line
// is used whole, and x is read in the same order of k. x goes through LDS in 128-deep
// chunks, double-buffered, shared by the waves; its 16-byte units are XORed with
// the row, which keeps the 16-row fragment reads free of bank conflicts. The weights of
// the next DEEP chunks are in flight while one is multiplied (4 KB a wave each), and with AHEAD the chunk's x beside
// them: loads come back in order, so that a wait for an x that was asked for last is one for all weights before it.
// (DEEP 4 up to 32 rows, 2 above: there x takes 16 registers a chunk. DEEP 4 without AHEAD does nothing. Us with x asked
// for one chunk before and so: 16384 x 2048 with silu 1 / 40 rows 19.2 / 22.6 and 18.2 / 19.6, 28672 x 4096 5 rows 52.2
// and 48.5, 8720 x 2048 in one share 15.6 and 12.3, 4096 x 14336 40 rows 27.9 and 25.9, 2048 x 2048 3.9 and 3.8. Above
// 64 rows the registers for it cost more workgroups than it gives: 28672 x 4096 120 rows 67 and 70.)
//
// A matrix of few rows is also split over k (linear_rows_splits); the splits' fp32 sums are left to the consumer, which reads them anyway (rope + store,
// residual + norm). Forms of the result:
//   PART  fp32 sums [S, M, N]          SILU  silu(gate) * up of a fused [gate; up] matrix
//   F32   fp32, S = 1 (logits)         CLAMPED  the clamped gated form of the hybrid family
//   BF16  rounded once, bias added before it
//
// Measured with the weights out of cache (the library's kernel in brackets), us:
//   4096 x 4096   5 rows 8.3 (15.6), 128 rows 15.6 (24.5)
//   4096 x 14336  5 rows 23.7 (26.7: 5 TB/s either way), 64 rows 28.7 (42), 128 rows 36 (75.5)
//   2048 x 8192   1 row 8.6 (12.8), 64 rows 11.4 (22.6)
//   28672 x 4096  with silu 48.5 (64 + 5) for 5 rows, 56 (54 + 5) for 64, 68 (57 + 5) for 128
// Above 64 rows every wave reads all of x from LDS for 16 weight rows, and LDS is the
// bound where K is not split far.

#include "common.h"

typedef __bf16 bf16x8_mfma __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

#define LR_KC 128          // k depth of a chunk
#define LR_STEPS 4         // matrix steps (32 k) of a chunk

enum LinearForm { LR_PART = 0, LR_BF16 = 1, LR_F32 = 2, LR_SILU = 3, LR_CLAMPED = 4 };

union LrFrag {
  u32x4 u;
  bf16x8_mfma m;
};

template <int MT, int FORM, int WAVES, int DEEP, bool AHEAD>
__global__ __launch_bounds__(64 * WAVES) void linear_rows_kernel(
    void* __restrict__ out, const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
    const bf16_t* __restrict__ bias, int M, int N, int K, int x_stride, int chunks_per_split, float limit, float alpha) {
  __shared__ __attribute__((aligned(16))) u32x4 xs[2][MT * 256];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int nchunks = K / LR_KC;
  const int c_begin = blockIdx.y * chunks_per_split;
  const int c_end = min(nchunks, c_begin + chunks_per_split);
  // weight row of this wave's tile; gated: the first half of the waves hold gate rows, the others the up rows of
  // the same columns
  constexpr int HW = WAVES / 2;
  constexpr bool GATED = FORM == LR_SILU || FORM == LR_CLAMPED;
  const int n0 = GATED ? (wave / HW) * (N / 2) + blockIdx.x * (16 * HW) + (wave % HW) * 16
                                 : blockIdx.x * (16 * WAVES) + wave * 16;
  const char* wrow = (const char*)(w + (int64_t)min(n0 + col, N - 1) * K) + grp * 32;

  f32x4 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};

  u32x4 wr[DEEP][LR_STEPS];
  constexpr int XP = MT * 4 / WAVES;      // passes of a chunk's x over the threads
  static_assert(XP >= 1, "as many 16-byte units as threads");
  constexpr int XD = AHEAD ? DEEP : 1;    // chunks of x in registers
  u32x4 xr[XD][XP];
  auto load_w = [&](int c, int slot, int st) {
    wr[slot][st] = *reinterpret_cast<const u32x4*>(wrow + (int64_t)c * (LR_KC * 2) + (st >> 1) * 128 + (st & 1) * 16);
  };
  // row tid / 16 of each pass, 16-byte unit tid % 16
  const int xrow = tid >> 4, xunit = tid & 15;
  auto load_x = [&](int c, int slot) {
#pragma unroll
    for (int i = 0; i < XP; ++i)
      xr[slot][i] = *reinterpret_cast<const u32x4*>((const char*)(x + (int64_t)min(i * 4 * WAVES + xrow, M - 1) * x_stride) +
                                              (int64_t)c * (LR_KC * 2) + xunit * 16);
  };
  auto store_x = [&](int buf, int slot) {
#pragma unroll
    for (int i = 0; i < XP; ++i) xs[buf][(i * 4 * WAVES + xrow) * 16 + (xunit ^ (xrow & 15))] = xr[slot][i];
  };

  if (c_begin < c_end) {
#pragma unroll
    for (int u = 0; u < DEEP; ++u)
      if (c_begin + u < c_end) {
        if (u < XD) load_x(c_begin + u, u);
#pragma unroll
        for (int st = 0; st < LR_STEPS; ++st) load_w(c_begin + u, u, st);
      }
    store_x(0, 0);
    __syncthreads();
    for (int c = c_begin; c < c_end; c += DEEP) {
#pragma unroll
      for (int u = 0; u < DEEP; ++u) {
        if (c + u < c_end) {
          const bool next = c + u + 1 < c_end;
          if (!AHEAD && next) load_x(c + u + 1, 0);
#pragma unroll
          for (int st = 0; st < LR_STEPS; ++st) {
            LrFrag a;
            a.u = wr[u][st];
#pragma unroll
            for (int i = 0; i < MT; ++i) {
              LrFrag b;
              b.u = xs[u & 1][i * 256 + col * 16 + (((st >> 1) * 8 + grp * 2 + (st & 1)) ^ col)];
              acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.m, b.m, acc[i], 0, 0, 0);
            }
          }
          if (c + u + DEEP < c_end) {
            if constexpr (AHEAD) load_x(c + u + DEEP, u);
#pragma unroll
            for (int st = 0; st < LR_STEPS; ++st) load_w(c + u + DEEP, u, st);
          }
          if (next) store_x(1 - (u & 1), (u + 1) % XD);
          __syncthreads();
        }
      }
    }
  }

  // lane (col, grp): rows n0 + grp*4 .. +3 of the weights, row i*16 + col of x
  const int n = n0 + grp * 4;
  if constexpr (GATED) {
    float* up = reinterpret_cast<float*>(&xs[0][0]);   // [HW waves][MT*16 rows][16]
    static_assert(HW * MT * 16 * 16 * 4 <= sizeof(xs), "the up halves fit the staging buffers");
    if (wave >= HW) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
        *reinterpret_cast<f32x4*>(up + (((wave - HW) * MT + i) * 16 + col) * 16 + grp * 4) = acc[i];
    }
    __syncthreads();
    if (wave < HW) {
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const int m = i * 16 + col;
        const f32x4 u = *reinterpret_cast<const f32x4*>(up + ((wave * MT + i) * 16 + col) * 16 + grp * 4);
        bf16x4_vec o;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if constexpr (FORM == LR_SILU) {
            // rounded as the separate product's result is
            const float g = bf16_to_f32(f32_to_bf16(acc[i][r])), v = bf16_to_f32(f32_to_bf16(u[r]));
            o[r] = f32_to_bf16(g / (1.0f + __expf(-g)) * v);
          } else {
            const float g = fminf(acc[i][r], limit), v = fminf(fmaxf(u[r], -limit), limit);
            o[r] = f32_to_bf16(g * (1.0f / (1.0f + expf(-alpha * g))) * (v + 1.0f));
          }
        }
        if (m < M) *reinterpret_cast<bf16x4_vec*>((short*)out + (int64_t)m * (N / 2) + n) = o;
      }
    }
  } else {
    if (n >= N) return;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int m = i * 16 + col;
      if (m >= M) continue;
      if constexpr (FORM == LR_PART) {
        *reinterpret_cast<f32x4*>((float*)out + ((int64_t)blockIdx.y * M + m) * N + n) = acc[i];
      } else if constexpr (FORM == LR_F32) {
        *reinterpret_cast<f32x4*>((float*)out + (int64_t)m * N + n) = acc[i];
      } else {
        bf16x4_vec o;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          o[r] = f32_to_bf16(acc[i][r] + (bias ? bf16_to_f32(((const short*)bias)[n + r]) : 0.0f));
        *reinterpret_cast<bf16x4_vec*>((short*)out + (int64_t)m * N + n) = o;
      }
    }
  }
}

// Waves of a workgroup. Eight halve the reads of x, which at 128 rows and 64 weight rows
// a workgroup are twice the weights' bytes; they pay where the weights still make enough
// workgroups. us with four and eight waves, weights out of cache:
//   PART, 65 / 96 / 128 rows   2048 x 2048  6.3 7.6 / 6.7 8.1 / 7.2 8.9     3072 x 2048  8.4 8.3 / 9.3 9.1 / 10.1 10.2
//     3072 x 8192  21.7 20.8 / 24.0 22.4 / 26.1 24.5     4096 x 4096  13.6 13.2 / 15.5 14.2 / 16.6 15.6
//     6144 x 4096  20.0 18.2 / 21.6 19.6 / 22.6 20.7     8192 x 8192  42.4 40.9 / 44.3 41.9 / 46.2 43.5
//   SILU, 33 / 64 rows   16384 x 2048  22.6 27.0 / 23.0 27.6     16384 x 4096  46.9 51.1 / 46.8 52.2
//     22016 x 4096  55.5 53.2 / 57.9 54.7     24576 x 3072  41.7 41.5 / 44.8 43.5     28672 x 4096  58.3 60.4 / 61.6 60.5
//   F32, 33 / 64 rows   16384 x 2048  21.8 26.3 / 22.4 27.6     24576 x 4096  53.6 54.3 / 57.1 56.6
//     50304 x 2048  56.9 52.0 / 61.3 54.5     128256 x 4096  217.9 220.3 / 240.5 232.5
// From 200 workgroups of eight waves on (N = 25600) neither side loses more than 4 %; a line at 20000 would gain the
// sizes between 3 - 6 %.
static int linear_rows_waves(int M, int N, int form) {
  if (N % 128 != 0) return 4;
  return (form == LR_PART ? M > 64 && N >= 4096 : M > 32 && N >= 200 * 128) ? 8 : 4;
}

extern "C" void launch_linear_rows(void* out, const bf16_t* x, const bf16_t* w, const bf16_t* bias, int M, int N,
                                   int K, int x_stride, int form, int splits, float limit, float alpha,
                                   hipStream_t stream) {
  const int per = (K / LR_KC + splits - 1) / splits;
  const int waves = linear_rows_waves(M, N, form);
  const dim3 grid((N + 16 * waves - 1) / (16 * waves), splits);
#define LR_GO(MT, F, WV, DEEP)                                                                                        \
  hipLaunchKernelGGL((linear_rows_kernel<MT, F, WV, DEEP, (MT <= 4)>), grid, dim3(64 * WV), 0, stream, out, x, w, bias, M, \
                     N, K, x_stride, per, limit, alpha)
#define LR_FORM(MT, WV, DEEP)                                \
  switch (form) {                                            \
    case LR_PART: LR_GO(MT, LR_PART, WV, DEEP); break;       \
    case LR_BF16: LR_GO(MT, LR_BF16, WV, DEEP); break;       \
    case LR_F32: LR_GO(MT, LR_F32, WV, DEEP); break;         \
    case LR_CLAMPED: LR_GO(MT, LR_CLAMPED, WV, DEEP); break; \
    default: LR_GO(MT, LR_SILU, WV, DEEP); break;            \
  }
  if (M <= 16) { LR_FORM(1, 4, 4); }
  else if (M <= 32) { LR_FORM(2, 4, 4); }
  else if (waves == 8 && M <= 64) { LR_FORM(4, 8, 2); }
  else if (waves == 8) { LR_FORM(8, 8, 2); }
  else if (M <= 64) { LR_FORM(4, 4, 2); }
  else { LR_FORM(8, 4, 2); }
#undef LR_FORM
#undef LR_GO
}

// splits of k for the PART form: about 800 workgroups, 512 (256 of eight waves) where
// the rows' sums weigh more (M > 32), and two chunks at least
extern "C" int linear_rows_splits(int M, int N, int K) {
  const int waves = linear_rows_waves(M, N, LR_PART);
  const int tiles = (N + 16 * waves - 1) / (16 * waves), chunks = K / LR_KC;
  int s = ((M <= 32 ? 800 : 2048 / waves) + tiles / 2) / tiles;
  s = s < chunks / 2 ? s : chunks / 2;
  return s < 1 ? 1 : s;
}
