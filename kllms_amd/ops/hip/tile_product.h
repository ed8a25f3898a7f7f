// The inner loop of the large bf16 products, for gfx950: a workgroup of 4 waves, one on
// each SIMD of a compute unit, multiplies 256 rows of W (columns of the result) with 32 * MJ rows of X,
// acc[i][j] of a wave = 16 columns i by 16 rows j of its 128 columns x 16 * MJ rows, in
// v_mfma_f32_16x16x32_bf16 (W the A operand, so that a lane ends with 4 neighbouring columns of a row).
//
// K goes by 64 ("stages") through a ring of LDS buffers, copied there straight from
// memory (no registers in between). Rows of 128 bytes; the copy writes LDS in lane
// order, so the conflict-free order of a row's 16-byte units (XORed with the row) is
// made by the addresses that the lanes read. A stage has two halves of 32 k:
//
//   first    matrix work on window 0 | window 1 is read to registers; barrier: the
//            buffer is free, the copy of stage s + RING into it starts
//   second   matrix work on window 1 | barrier before it: stage s + 1 has landed; its
//            window 0 is read, the copy goes on
//
// What bounds it: the matrix units, and around them the issue of the copies. A copy
// instruction of 1 KB occupies the address unit for 16 cycles; issued in bursts the
// waves stall on it (1319 TFLOP/s at 8192^3), spread evenly over a stage, one every 5
// matrix instructions, it stays under them (1490, where the library reaches 1570; 1260
// with half as deep stages of 64-byte rows, whose requests are twice as many; 1360 with
// 32x32x16 instructions). The order of issue is pinned by scheduling barriers.
// One wave per SIMD (128 x 128 of the result) needs 1.0 KB of LDS reads per 4 matrix instructions, half of
// what eight waves of 128 x 64 need, and all 512 registers: 256 sums, 2 x 64 fragments.
//
// Small MJ are for the ends of ragged row ranges and for few rows, where the stream of W
// is the bound: less matrix work per stage, and more buffers of it in flight. So are NI of 2 and 4, tiles of 64 and 128
// rows of W for products that it bounds from end to end (linear_rows.hip). One loop for all of their stages: with the last
// ones in a loop of their own, without copies, the sums moved between registers in every stage (28672 x 4096, 256 rows:
// 82 us; 64 so).

#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.h"

typedef __bf16 bf16x8_mfma __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_cvt __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

#define TP_N 256           // rows of W of a workgroup
#define TP_K 64            // k of a stage
#define TP_THREADS 256
#define TP_LDS 163840      // all of a compute unit's
#define TP_SLOTS 32        // compute units of an XCD
#define TP_SHARES 4        // workgroups that share a tile's K at most
#define TP_SUMS (256 * 256)

// Which of an XCD's tiles its at-th workgroup takes, and which share of its K. Tiles that
// make whole rounds of the XCD's compute units are one workgroup's each; those of the
// last round, if they leave half of the units idle or more, are shared out.
struct TileShare {
  int tile, share, shares;
  float* part;               // [8 XCDs][TP_SLOTS][sums], of this tile's shares; sums: floats of a tile at most
  int* count;                // [8][TP_SLOTS] zeros
  __device__ __forceinline__ TileShare(int at, int tiles, int stages, float* parts, int* counts, int xcd,
                                       int sums = TP_SUMS)
      : tile(at), share(0), shares(1), part(nullptr), count(nullptr) {
    const int rest = tiles % TP_SLOTS, full = tiles - rest;
    if (!parts || at < full || rest == 0) return;
    shares = max(1, min(min(TP_SLOTS / rest, TP_SHARES), stages / 8));
    const int r = (at - full) % rest;
    share = (at - full) / rest;
    tile = share < shares ? full + r : tiles;
    part = parts + (int64_t)(xcd * TP_SLOTS + r * shares) * sums;
    count = counts + xcd * TP_SLOTS + r;
  }
  __device__ __forceinline__ int first(int stages) const { return (stages + shares - 1) / shares * share; }
  __device__ __forceinline__ int length(int stages) const {
    return min((stages + shares - 1) / shares, stages - first(stages));
  }
};

#define TP_HOLD __builtin_amdgcn_sched_barrier(0)

// Buffer descriptor of bytes from p on; lanes whose own offset is behind its end read zeros.
__device__ __forceinline__ u32x4 tp_range(const void* p, uint32_t bytes) {
  const uint64_t a = (uint64_t)p;
  u32x4 r;
  r[0] = __builtin_amdgcn_readfirstlane((uint32_t)a);
  r[1] = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32)) & 0xffff;
  r[2] = __builtin_amdgcn_readfirstlane(bytes);
  r[3] = 0x00020000;
  return r;
}

// Copies of 16 bytes a lane to lds + lane * 16. They are written out because the
// compiler makes every later LDS read wait for the builtin's; the waits stand in the loop.
// The step to the copy's row is in the lane's offset, which the range check covers: of the scalar offset it
// only has to hold that it stays within the range (k inside a row), not what a check makes of one beyond it.
// ONCE: the caches need not hold it for longer than it takes (nt).
template <bool ONCE = false>
__device__ __forceinline__ void tp_copy(u32x4 range, uint32_t lane_off, uint32_t off, uint32_t lds) {
  if constexpr (ONCE)
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen nt lds" ::"v"(lane_off), "s"(range),
                 "s"(off), "s"(lds)
                 : "memory");
  else
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(lane_off), "s"(range),
                 "s"(off), "s"(lds)
                 : "memory");
}

__device__ __forceinline__ void tp_copy_at(uint64_t at, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(at), "s"(lds) : "memory");
}

// Rows of an operand in memory order, 8 to a copy: from row ``first`` of p on, those before ``end`` (1 or more) and
// ``most`` of them at most; the others read as zeros. Behind the end altogether the last row stands in, so that the
// range always holds a row: what comes of it belongs to rows or columns that are not stored. K: elements from a row to the
// next, width: those of a row that are read. The range ends with the last row's: rows may overlap or be one and the same
// (K below width), and then what does not exist reads others' values, for rows that are not stored either.
template <bool ONCE>
struct TileRowsOf {
  u32x4 range;
  uint32_t at[8];            // this lane's offset in each copy: the same registers for all operands of one K
  __device__ __forceinline__ TileRowsOf(const bf16_t* p, int first, int end, int most, int K, int lane)
      : TileRowsOf(p, first, end, most, K, K, lane) {}
  __device__ __forceinline__ TileRowsOf(const bf16_t* p, int first, int end, int most, int K, int width, int lane)
      : range(tp_range(p + (int64_t)min(first, end - 1) * K,
                       ((uint32_t)(min(end - min(first, end - 1), most) - 1) * K + width) * 2)) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      at[i] = (uint32_t)(i * 8 + (lane >> 3)) * K * 2 + (((lane & 7) ^ (lane >> 3)) << 4);
  }
  __device__ __forceinline__ void copy(int i, uint32_t k_off, uint32_t lds) const { tp_copy<ONCE>(range, at[i], k_off, lds); }
  // zeros, without a look at memory, where not ``live``
  __device__ __forceinline__ void copy(int i, uint32_t k_off, uint32_t lds, bool live) const {
    u32x4 r = range;
    r[2] = live ? r[2] : 0;
    tp_copy<ONCE>(r, at[i], k_off, lds);
  }
};
typedef TileRowsOf<false> TileRows;

// Rows anywhere: at[i] is the address of this lane's 16 bytes of the i-th copy in stage 0.
template <int MJ>
struct TileGather {
  uint64_t at[MJ];
  __device__ __forceinline__ void copy(int i, uint32_t k_off, uint32_t lds) const { tp_copy_at(at[i] + k_off, lds); }
};

template <int MJ, int NI = 8, int BYTES = TP_LDS>
struct TileRing {
  static constexpr int STRIDE = (32 * NI + 32 * MJ) * 128;   // W rows, then X rows
  static constexpr int MOST = NI == 8 ? 4 : 8;
  static constexpr int RING = BYTES / STRIDE < MOST ? BYTES / STRIDE : MOST;
};

// acc += W X^T over K; w: this wave's 8 * NI of the 32 * NI rows (64 of 256), x: its 8 * MJ of the 32 * MJ. Ends with all
// waves past their last LDS read. NI 4, tiles of 128 columns, is for few rows: half the sums, more buffers in flight.
template <int MJ, int NI = 8, int BYTES = TP_LDS, class W, class X>
__device__ __forceinline__ void tile_product(f32x4 (&acc)[NI][MJ], const W& w, const X& x, int stages, int start,
                                             char* smem) {
  constexpr int STRIDE = TileRing<MJ, NI, BYTES>::STRIDE, RING = TileRing<MJ, NI, BYTES>::RING;
  constexpr int G = NI * MJ;             // matrix instructions of a half
  constexpr int NR = NI + MJ;            // LDS reads of a half
  constexpr int ND = NI + MJ;            // copies of a stage
  constexpr int F = G > NR + 3 ? G : NR + 3;   // places for them, the reads and the copies
  constexpr int BOTH = NI < MJ ? NI : MJ;   // reads and copies go by turns while both operands have some
  constexpr int RS = F / (2 * NR) > 0 ? F / (2 * NR) : 1;
  constexpr int P1 = RS * NR + (NI < 8 ? (F - RS * NR) / 2 : MJ >= 4 ? 8 : 4);   // first half: all has been read
  constexpr int DS = (2 * F - P1) / ND;             // a copy every DS instructions from there on
  constexpr int D1 = (F - 1 - P1) / DS + 1;         // copies in the first half
  constexpr bool LEAN = NI < 8;          // few stages: what is behind the last is out of the copies' range, and not read
  static_assert(P1 < F && DS >= 1 && RING >= 2 && (RING - 1) * ND < 64);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  const uint32_t w_put = lds0 + wave * NI * 1024, x_put = lds0 + NI * 4096 + wave * MJ * 1024;
  uint32_t w_get[2], x_get[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const uint32_t o = lds0 + col * 128 + (((ks * 4 + grp) ^ (col & 7)) << 4);
    w_get[ks] = o + (wave >> 1) * NI * 16 * 128;
    x_get[ks] = o + NI * 4096 + (wave & 1) * MJ * 16 * 128;
  }
  typedef __attribute__((address_space(3))) const bf16x8_mfma* lds_ptr;
  auto get = [](uint32_t at) { return *(lds_ptr)(uintptr_t)at; };
  bool live = true;                      // the stage that is copied exists
  auto put = [&](int d, uint32_t k_off, uint32_t buf) {   // d-th copy of a stage
    const int i = d < 2 * BOTH ? d >> 1 : d - BOTH;
    if constexpr (LEAN) {
      if (d < 2 * BOTH ? d & 1 : MJ > NI) x.copy(i, k_off, x_put + buf + i * 1024, live);
      else w.copy(i, k_off, w_put + buf + i * 1024, live);
    } else {
      if (d < 2 * BOTH ? d & 1 : MJ > NI) x.copy(i, k_off, x_put + buf + i * 1024);
      else w.copy(i, k_off, w_put + buf + i * 1024);
    }
  };
  auto k_at = [&](int t) {               // of the t-th stage in work; behind the last one, that one's
    const int i = min(t, stages - 1) + start;
    return (uint32_t)(i < stages ? i : i - stages) * 128;
  };
  bf16x8_mfma a[2][NI], b[2][MJ];
  auto read = [&](int ks, int r, uint32_t buf) {
    const int i = r < 2 * BOTH ? r >> 1 : r - BOTH;
    if (r < 2 * BOTH ? !(r & 1) : MJ > NI) b[ks][i] = get(x_get[ks] + buf + i * 2048);
    else a[ks][i] = get(w_get[ks] + buf + i * 2048);
  };
  auto multiply = [&](int ks, int f) {
    if (f >= G) return;
    const int i = f / MJ, j = f % MJ;
    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ks][i], b[ks][j], acc[i][j], 0, 0, 0);
    if (f & 1) TP_HOLD;
  };

#pragma unroll
  for (int t = 0; t < RING; ++t) {       // of fewer stages the last one again: the counts below stand
    live = t < stages;
#pragma unroll
    for (int d = 0; d < ND; ++d) put(d, k_at(t), t * STRIDE);
  }
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"((RING - 1) * ND) : "memory");
#pragma unroll
  for (int r = 0; r < NR; ++r) read(0, r, 0);

  uint32_t buf = 0;
#pragma unroll 1
  for (int s = 0; s < stages; ++s) {
    // behind the last stage that one is copied again and nothing of it used: no branches
    const uint32_t k_off = k_at(s + RING);
    live = s + RING < stages;
    TP_HOLD;
#pragma unroll
    for (int f = 0; f < F; ++f) {
      if (f % RS == 0 && f / RS < NR) read(1, f / RS, buf);
      if (f == P1) {
        __builtin_amdgcn_s_waitcnt(0xC07F);           // lgkmcnt(0)
        asm volatile("s_barrier" ::: "memory");
        TP_HOLD;
      }
      if (f >= P1 && (f - P1) % DS == 0 && (f - P1) / DS < ND) put((f - P1) / DS, k_off, buf);
      multiply(0, f);
    }
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"((RING - 2) * ND + D1) : "memory");
    TP_HOLD;
    const uint32_t next = buf == (RING - 1) * STRIDE ? 0u : buf + STRIDE;
#pragma unroll
    for (int f = 0; f < F; ++f) {
      if (f % RS == 0 && f / RS < NR) read(0, f / RS, next);
      if ((f + F - P1) % DS == 0 && (f + F - P1) / DS < ND) put((f + F - P1) / DS, k_off, buf);
      multiply(1, f);
    }
    buf = next;
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  // what follows reads sums out of the accumulation registers; it is held off the loop, which must not move them
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j) asm volatile("" : "+a"(acc[i][j]));
}

// Sums of a tile whose K is shared by ``shares`` workgroups: each leaves its own in part
// [shares][8 * MJ][threads][4]; the last one to arrive adds them all up, in the order
// of the shares whoever it is, and goes on (true) with the whole. count: 0 before.
//
// The sums are stored past the XCD's L2 and read past it (sc1), and each wave waits for its stores before the count. A
// fence of the device's scope instead writes back and invalidates that whole L2, under everybody who works on it. 2048
// columns, K 8192, in up to four shares of 64-row tiles: 150 rows 52 us with the fences, 33 without; 700 rows 70 and 47.
template <int MJ>
__device__ __forceinline__ bool tile_fold(f32x4 (&acc)[8][MJ], float* part, int share, int shares, int* count, char* smem) {
  constexpr int SIZE = 8 * MJ * TP_THREADS * 16, SC1 = 16;
  const int tid = threadIdx.x;
  const auto all = __builtin_amdgcn_make_buffer_rsrc(part, 0, shares * SIZE, 0x00020000);
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[i][j]), all, tid * 16,
                                            share * SIZE + (i * MJ + j) * TP_THREADS * 16, SC1);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0)
    *reinterpret_cast<int*>(smem) = __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (*reinterpret_cast<const int*>(smem) != shares - 1) return false;
  __syncthreads();                       // smem is free again
  // 32 loads of a thread at a time
#pragma unroll
  for (int i0 = 0; i0 < 8; i0 += 2) {
    f32x4 sum[2][MJ];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < MJ; ++j) sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int s0 = 0; s0 < shares; s0 += 2) {
      u32x4 v[2][2][MJ];
      auto load = [&](int e) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < MJ; ++j)
            v[e][i][j] = __builtin_amdgcn_raw_buffer_load_b128(all, tid * 16, (s0 + e) * SIZE + ((i0 + i) * MJ + j) * TP_THREADS * 16, SC1);
      };
      load(0);
      if (s0 + 1 < shares) {
        load(1);
      } else {                           // an odd number of shares: the last one alone, nothing is read behind it
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < MJ; ++j) v[1][i][j] = u32x4{0u, 0u, 0u, 0u};
      }
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < MJ; ++j) {
            const f32x4 x = __builtin_bit_cast(f32x4, v[e][i][j]);
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[i][j][r] += x[r];
          }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < MJ; ++j) acc[i0 + i][j] = sum[i][j];
    TP_HOLD;
  }
  return true;
}

__device__ __forceinline__ bf16x4_vec tp_pack(float a, float b, float c, float d) {
  const f32x4 v = {a, b, c, d};
  return __builtin_bit_cast(bf16x4_vec, __builtin_convertvector(v, bf16x4_cvt));
}

// A wave's result, 16 * MJ rows by 16 * NI columns, to memory in 16-byte stores of whole rows, by way of its own part
// of LDS: value(i, j) gives the lane's 4 columns i * 16 + grp * 4.. of row j * 16 + col. Row r goes to out + r *
// stride; rows and columns of it exist, columns and stride are multiples of 8.
template <int NI, int MJ, class V>
__device__ __forceinline__ void tile_store(bf16_t* out, int64_t stride, int rows, int columns, char* smem, V value) {
  constexpr int UNITS = NI * 2;          // 16-byte units of a row: 4, 8 or 16
  const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
  char* mine = smem + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * (MJ * 16 * UNITS * 16);
#pragma unroll
  for (int j = 0; j < MJ; ++j)
#pragma unroll
    for (int i = 0; i < NI; ++i)
      *reinterpret_cast<bf16x4_vec*>(mine + (j * 16 + col) * (UNITS * 16) +
                                     (((i * 2 + (grp >> 1)) ^ (col & (UNITS - 1))) << 4) + (grp & 1) * 8) = value(i, j);
  // this wave's own part of LDS: in order, only the compiler is held
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const int unit = lane % UNITS, r0 = lane / UNITS;
#pragma unroll
  for (int k = 0; k < MJ * 16 * UNITS / 64; ++k) {
    const int r = k * (64 / UNITS) + r0;
    const u32x4 v = *reinterpret_cast<const u32x4*>(mine + r * (UNITS * 16) + ((unit ^ (r & (UNITS - 1))) << 4));
    if (r < rows && unit * 8 < columns) *reinterpret_cast<u32x4*>((short*)out + r * stride + unit * 8) = v;
  }
}

// room for all of LDS, asked for at each launch: the attribute is the current device's
static inline bool tp_lds_ready(const void* kernel) {
  return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, TP_LDS) == hipSuccess;
}
