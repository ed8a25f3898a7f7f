// Sampling + logprob for gfx950, in two launches (one for short rows).
//
//   sample_part   every row cut into slices, one 256-thread workgroup each: the
//                 slice's max and argmax, its sum of exp, and - for rows
//                 without top-p / top-k - the Gumbel-max draw over the slice
//   sample_final  one workgroup per row: folds the slices; rows with top-p /
//                 top-k find their threshold and draw here
//
// Why split: one workgroup per row leaves a 120-row batch on 120 of 256 compute
// units and a 16-row one on 16, and walks the row three times. Arithmetic, not
// memory, bounds the split form: per token the hash in 32-bit products, two
// logarithms, the exponential of the sum and the compares, 28 us for 120 x 128256
// tokens where greedy rows take 17 (the logits alone: 61.6 MB, 13 us at the 4.7 TB/s
// a copy reaches), 35 where all rows are truncated and listed instead of drawn.
//
// Rows with top-p / top-k: each slice of a long row lists its highest tokens (slice_list), and sample_final finds the
// cut in the lists alone where they reach it. It counts their scaled mass and number in 256 bins (per-wave copies: a
// single one serialises on same-bin LDS atomics), which names the boundary bin, and up to 3 refinements at 256x finer
// resolution each (20/256^4 ~ 5e-9 in scaled-logit space: exact up to fp32 rounding of the logits) the threshold in it.
// Rows whose cut lies behind the lists, and rows without any, are swept by their one workgroup: atomics and exponentials
// are what a sweep costs, so the bins near the max are counted first, with their tokens listed in LDS; flat rows take
// further sweeps, and a boundary bin that outgrows the list is refined by rescans of the row.
//
// Measured, 128256 tokens a row: 120 rows, half of them with top-p 0.95 and top-k 50, 50 us (79 with sweeps alone, 346 with
// one workgroup per row walking it three to six times); 8 rows, all truncated, 24 us (52). With the draw of slice_part:
// 43.7 us for the 120 rows, 8.8 us for 16 masked ones. With lists that each thread places its own tokens in (by ballots and
// a counter in LDS 8.6 us of a slice's 22, now 4.4 of 16) and the cut made from tokens in registers (12 us a row, now 8):
// 36 us for the 120 rows, 17 for 7 truncated ones.
//
// The draw is counter-based: hash(seed, step, token), identical regardless of
// batch composition and of the slicing. What follows from a sum is so to fp32
// rounding only, since the slices of a row depend on the rows beside it:
// log-probabilities, and the mass at which top-p cuts (about 1e-7 of the row's; a
// token whose share ends within that of top_p may be in at one batch size and out at
// another). Slices by V alone cost up to 20% (250 rows of 152064: 75 us -> 90).
// temperature == 0 -> greedy.

#include <type_traits>

#include "common.h"

// sx(x) must be BIT-IDENTICAL across the histogram, the refinements and the
// admission. hipcc contracts even
// __fmul_rn/__fsub_rn pairs into an fma, and may do so at one site but not
// another — the recomputed sx of the MAX token then comes out as the
// product's rounding residual (~1e-10, either sign) instead of 0 and falls
// outside the (lo, 0] boundary interval (observed: the max missing from the
// refinement histogram on half the rows -> k+1 admitted). ONE explicit fma
// is a single IR op the compiler cannot split or re-associate, so every
// pass computes the same bits.
__device__ __forceinline__ float sx_of(float x, float inv_t, float smax) {
  return __builtin_fmaf(x, inv_t, -smax);
}

#define NT 1024
#define NW (NT / WAVE)     // 16 waves
#define SBINS 256
#define SRANGE 20.0f       // scaled-logit window below max covered by the histogram
// bins counted by the first, second and third sweep: scaled logits within 5 of
// the max, within 10, the rest. A sweep that counts every token is bound by its
// two LDS atomics (about one lane a cycle: 100 us for 128k tokens), one that counts
// a few hundred by its loads (8 us); most rows' cut lies within 10
#define SNEAR 64
#define SMID 128
#define SLIST 3072         // tokens listed in LDS (a flat row of 128k tokens has up to ~2500 in its boundary bin)
#define PT 256             // threads of a slice's workgroup
#define PU 8               // logits in flight per thread

// what a slice hands to sample_final: 10 words
struct SlicePart {
  float max;
  float sum;                 // sum of exp(x - max)
  int arg;                   // lowest token at the max, -1: none above -inf
  float ssum;                // rows with top-p / top-k: sum of exp((x - max) / temperature)
  unsigned long long best;   // ordered key bits << 32 | token
  float edge;                // rows with top-p / top-k: the slice's tokens from this logit on are in its list; inf: none
  int listed;                // how many they are
  float mass;                // and their sum of exp((x - max) / temperature)
  int unused;
};

struct SliceToken { float x; int tok; };

__device__ __forceinline__ unsigned long long pack_key(float key, int tok) {
  uint32_t k = __float_as_uint(key);
  k = (k & 0x80000000u) ? ~k : (k | 0x80000000u);
  return ((unsigned long long)k << 32) | (uint32_t)tok;
}

// key bits of -inf: nothing was drawn
#define NO_KEY 0x007fffffu

__device__ __forceinline__ uint64_t draw_base(int64_t seed, int64_t step) {
  return splitmix64((uint64_t)seed * 0x9E3779B97F4A7C15ULL + (uint64_t)step * 0xBF58476D1CE4E5B9ULL);
}

// splitmix64 of a row's base ^ token, the upper word without its last step, which leaves the 24 bits that are used as they
// are. What of it is the row's alone is worked out once: the upper half of the first sum has two values, by the carry.
// In words of 32 bits: a shift of 64 issues at a fraction of the rate
struct Draw {
  uint32_t lo, hi;           // of the base, the upper half with the constant added
  uint32_t far0, far1;       // product of the mixed upper half without and with a carry
  float inv_t;
  __device__ __forceinline__ Draw(uint64_t base, float inv)
      : lo((uint32_t)base), hi((uint32_t)(base >> 32) + 0x9E3779B9u), inv_t(inv) {
    far0 = (hi ^ (hi >> 30)) * 0x1CE4E5B9u;
    far1 = ((hi + 1) ^ ((hi + 1) >> 30)) * 0x1CE4E5B9u;
  }
  __device__ __forceinline__ uint32_t word(int tok) const {
    const uint32_t s = (lo ^ (uint32_t)tok) + 0x7F4A7C15u;
    const bool carry = s < 0x7F4A7C15u;
    const uint32_t a = s ^ __builtin_amdgcn_alignbit(hi + carry, s, 30);
    const uint64_t p = (uint64_t)a * 0x1CE4E5B9u;
    uint32_t ph = (uint32_t)(p >> 32) + a * 0xBF58476Du + (carry ? far1 : far0);
    const uint32_t pl = (uint32_t)p ^ __builtin_amdgcn_alignbit(ph, (uint32_t)p, 27);
    ph ^= ph >> 27;
    return __umulhi(pl, 0x133111EBu) + pl * 0x94D049BBu + ph * 0x133111EBu;
  }
  __device__ __forceinline__ float key(int tok, float x) const {
    const float u = (float)((word(tok) >> 8) + 1) * (1.0f / 16777217.0f);   // (0, 1]
    const float gumbel = -__logf(-__logf(u));
    return x * inv_t + gumbel;
  }
  // key up to rounding: the logarithms as the hardware has them
  __device__ __forceinline__ float near(int tok, float x) const {
    constexpr float LN2 = 0.693147180559945309f;
    const float u = (float)((word(tok) >> 8) + 1) * (1.0f / 16777217.0f);
    return __builtin_fmaf(x, inv_t, -LN2 * __builtin_amdgcn_logf(-LN2 * __builtin_amdgcn_logf(u)));
  }
};

__device__ __forceinline__ bool truncates(float top_p, int top_k, int V) {
  return (top_p < 1.0f) || (top_k > 0 && top_k < V);
}

// exp(a - m) with exp(-inf - -inf) taken as an empty sum
__device__ __forceinline__ float exp_from(float a, float m) {
  return a == -INFINITY ? 0.0f : __expf(a - m);
}

__device__ __forceinline__ unsigned long long wave_max_u64(unsigned long long v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const unsigned long long o = __shfl_xor(v, off);
    v = o > v ? o : v;
  }
  return v;
}

// op over the wave's 64 values, in all lanes, without a trip through LDS: all lanes take part
template <class T, class Op>
__device__ __forceinline__ T wave_fold(T v, Op op) {
  auto bits = [](T x) { return __builtin_bit_cast(int, x); };
  auto back = [](int x) { return __builtin_bit_cast(T, x); };
  v = op(v, back(__builtin_amdgcn_mov_dpp(bits(v), 0xB1, 0xf, 0xf, false)));    // neighbours
  v = op(v, back(__builtin_amdgcn_mov_dpp(bits(v), 0x4E, 0xf, 0xf, false)));    // pairs of a quad
  v = op(v, back(__builtin_amdgcn_mov_dpp(bits(v), 0x141, 0xf, 0xf, false)));   // quads of 8
  v = op(v, back(__builtin_amdgcn_mov_dpp(bits(v), 0x140, 0xf, 0xf, false)));   // halves of a row of 16
  const auto rows = __builtin_amdgcn_permlane16_swap((unsigned)bits(v), (unsigned)bits(v), false, false);
  v = op(back((int)rows[0]), back((int)rows[1]));
  const auto halves = __builtin_amdgcn_permlane32_swap((unsigned)bits(v), (unsigned)bits(v), false, false);
  return op(back((int)halves[0]), back((int)halves[1]));
}

// sums up to and with each lane, likewise: shifts in rows of 16, then the rows' ends to the rows behind them
template <class T>
__device__ __forceinline__ T wave_scan(T v) {
  auto bits = [](T x) { return __builtin_bit_cast(int, x); };
  auto back = [](int x) { return __builtin_bit_cast(T, x); };
  v += back(__builtin_amdgcn_update_dpp(0, bits(v), 0x111, 0xf, 0xf, false));
  v += back(__builtin_amdgcn_update_dpp(0, bits(v), 0x112, 0xf, 0xf, false));
  v += back(__builtin_amdgcn_update_dpp(0, bits(v), 0x114, 0xf, 0xf, false));
  v += back(__builtin_amdgcn_update_dpp(0, bits(v), 0x118, 0xf, 0xf, false));
  v += back(__builtin_amdgcn_update_dpp(0, bits(v), 0x142, 0xa, 0xf, false));
  v += back(__builtin_amdgcn_update_dpp(0, bits(v), 0x143, 0xc, 0xf, false));
  return v;
}

// the lane before's value, 0 in the first
template <class T>
__device__ __forceinline__ T wave_before(T v) {
  return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x138, 0xf, 0xf, false));
}

// tokens [lo, hi) of a row by a workgroup of THREADS, lo a multiple of 64; the result is thread 0's. strip: room for the tokens of a masked row
// that are allowed, PU * 64 a wave, or nullptr.
//
// The draw: what bounds a slice is the issue of its arithmetic, and the hash alone is half of that. So a token's key is not
// worked out to the last bit (two logarithms with their corrections are a third of it); a lane keeps its highest and
// second highest key up to rounding. The exact key is made for the highest of each lane; where it then is not clear that
// no lane's second one can win, the wave makes all of its keys. The draw is so the same to the last bit as with all keys.
// Of a masked row the allowed tokens are packed first, so that waves work on 64 of them at a time, and the mask is read a
// word for 32 lanes. us with all keys made and now, masked with one token in eight allowed in brackets: 120 rows of 128256
// 38.9, 29.2 (44.9, 20.4)   16 rows 11.5, 10.0 (12.1, 8.8)   250 rows of 152064 74.5, 56.8 (90.3, 36.6); 120 greedy rows take 17.
template <int THREADS>
__device__ __forceinline__ SlicePart slice_part(const float* __restrict__ row, const uint32_t* __restrict__ mrow,
                                                float temp, bool cuts, uint64_t base, int lo, int hi,
                                                SliceToken* __restrict__ strip) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool draw = temp != 0.0f && !cuts;
  const float inv_t = (temp > 0.0f) ? 1.0f / temp : 0.0f;

  float m = -INFINITY, sum = 0.0f, ssum = 0.0f;
  float first = -INFINITY, second = -INFINITY;     // highest keys
  int arg = -1, at = -1;
  const Draw rng(base, inv_t);
  auto consider = [&](int tok, float x) {          // -inf and NaN change nothing
    const float v = rng.near(tok, x);
    if (v > first) at = tok;
    second = __builtin_amdgcn_fmed3f(second, first, v);
    first = fmaxf(first, v);
  };
  auto higher = [&](float cm) {
    sum *= exp_from(m, cm);
    ssum *= m == -INFINITY ? 0.0f : __expf((m - cm) * inv_t);
    m = cm;
  };
  // the wave's allowed tokens among the 64 from i0 + j * THREADS on, for all j: whole words of the mask, the same for all
  // lanes (lo is a multiple of 64)
  auto allowed = [&](int i0, auto whole, uint64_t (&votes)[PU]) {
    const uint32_t* words = mrow + (i0 >> 5);
#pragma unroll
    for (int j = 0; j < PU; ++j) {
      if constexpr (whole()) {
        votes[j] = words[j * (THREADS / 32)] | (uint64_t)words[j * (THREADS / 32) + 1] << 32;
      } else {
        const int n = max(min(hi - (i0 + j * THREADS), 64), 0);
        votes[j] = n == 0 ? 0 : (words[j * (THREADS / 32)] | (n > 32 ? (uint64_t)words[j * (THREADS / 32) + 1] << 32 : 0)) & ~0ull >> (64 - n);
      }
    }
  };
  // a wave's lanes stay together: 64 tokens from i0 on, and from each THREADS behind
  auto round = [&](int i0, auto whole) {
    float x[PU];
    const float* from = row + i0;
#pragma unroll
    for (int j = 0; j < PU; ++j) x[j] = from[whole() ? j * THREADS + lane : min(j * THREADS + lane, hi - 1 - i0)];
    uint64_t votes[PU];
    if (mrow) allowed(i0, whole, votes);
    if (mrow && strip) {
      SliceToken* mine = strip + wave * (PU * WAVE);
      int n = 0;
#pragma unroll
      for (int j = 0; j < PU; ++j) {
        if (__builtin_amdgcn_inverse_ballot_w64(votes[j]))
          mine[n + __builtin_amdgcn_mbcnt_hi((uint32_t)(votes[j] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)votes[j], 0))] =
              SliceToken{x[j], i0 + j * THREADS + lane};
        n += (int)__popcll(votes[j]);
      }
      // the strip is this wave's own: in-order LDS, only the compiler is held
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      for (int e0 = 0; e0 < n; e0 += WAVE) {
        const SliceToken t = mine[min(e0 + lane, n - 1)];
        const float v = e0 + lane < n ? t.x : -INFINITY;
        if (v > m) {
          higher(v);
          arg = t.tok;
        }
        sum += exp_from(v, m);
        if (cuts && v != -INFINITY) ssum += __expf((v - m) * inv_t);
        if (draw) consider(t.tok, v);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      return;
    }
    if (mrow) {
#pragma unroll
      for (int j = 0; j < PU; ++j) x[j] = __builtin_amdgcn_inverse_ballot_w64(votes[j]) ? x[j] : -INFINITY;
    } else if (!whole()) {
#pragma unroll
      for (int j = 0; j < PU; ++j) x[j] = i0 + j * THREADS + lane < hi ? x[j] : -INFINITY;
    }
    float cm = x[0];
#pragma unroll
    for (int j = 1; j < PU; ++j) cm = fmaxf(cm, x[j]);
    if (cm > m) {
      higher(cm);
#pragma unroll
      for (int j = PU - 1; j >= 0; --j)
        if (x[j] == cm) arg = i0 + j * THREADS + lane;
    }
    const float near = m == -INFINITY ? 0.0f : m;  // -inf adds nothing, also before a finite token
#pragma unroll
    for (int j = 0; j < PU; ++j) sum += __expf(x[j] - near);
    if (cuts) {
#pragma unroll
      for (int j = 0; j < PU; ++j)
        if (x[j] != -INFINITY) ssum += __expf((x[j] - m) * inv_t);
    }
    if (draw) {
#pragma unroll
      for (int j = 0; j < PU; ++j) consider(i0 + j * THREADS + lane, x[j]);
    }
  };
  int i0 = lo + wave * WAVE;
  for (; i0 + THREADS * (PU - 1) + WAVE <= hi; i0 += THREADS * PU) round(i0, std::true_type{});
  if (i0 < hi) round(i0, std::false_type{});

  auto most = [](float a, float b) { return fmaxf(a, b); };
  auto plus = [](float a, float b) { return a + b; };
  float best = -INFINITY;
  if (draw) {
    if (at >= 0) {
      const float key = rng.key(at, row[at]);
      if (key > best) best = key;
    }
    const float top = wave_fold(best, most);
    // an infinite key (u of one) is so in both forms
    const bool open = second != -INFINITY && (top == INFINITY ? second == top : !(second < top - (1e-3f + 1e-6f * fabsf(top))));
    if (__any(open) || (top != -INFINITY && __popcll(__ballot(best == top)) > 1)) {
      best = -INFINITY;
      for (int i0 = lo + wave * WAVE; i0 < hi; i0 += THREADS * PU) {
        float x[PU];
        uint64_t votes[PU];
#pragma unroll
        for (int j = 0; j < PU; ++j) x[j] = row[min(i0 + j * THREADS + lane, hi - 1)];
        if (mrow) allowed(i0, std::false_type{}, votes);
#pragma unroll
        for (int j = 0; j < PU; ++j) {
          const int tok = i0 + j * THREADS + lane;
          const bool ok = mrow ? (votes[j] >> lane & 1) != 0 : tok < hi;
          const float key = rng.key(tok, x[j]);
          if (ok && key > best) { best = key; at = tok; }
        }
      }
    }
  }

  // fold the lanes, then the waves: max, lowest token at it, rescaled sums, best key
  __shared__ float sh_m[THREADS / WAVE], sh_s[THREADS / WAVE], sh_ss[THREADS / WAVE], sh_key[THREADS / WAVE];
  __shared__ int sh_tok[THREADS / WAVE], sh_arg[THREADS / WAVE];
  const float M = wave_fold(m, most);
  const float S = wave_fold(sum * (m == M ? 1.0f : exp_from(m, M)), plus);
  const float SS = cuts ? wave_fold(ssum * (m == M ? 1.0f : m == -INFINITY ? 0.0f : __expf((m - M) * inv_t)), plus) : 0.0f;
  const int a = wave_fold((m == M && arg >= 0) ? arg : 0x7fffffff, [](int p, int q) { return min(p, q); });
  const float K = wave_fold(best, most);
  const int tok = wave_fold(best == K ? at : -1, [](int p, int q) { return max(p, q); });   // of equal keys the last token
  if (lane == 0) {
    sh_m[wave] = M;
    sh_s[wave] = S;
    sh_ss[wave] = SS;
    sh_arg[wave] = a;
    sh_key[wave] = K;
    sh_tok[wave] = tok;
  }
  __syncthreads();
  SlicePart p;
  if (tid == 0) {
    p.max = sh_m[0];
#pragma unroll
    for (int k = 1; k < THREADS / WAVE; ++k) p.max = fmaxf(p.max, sh_m[k]);
    p.sum = p.ssum = 0.0f;
    p.arg = 0x7fffffff;
    p.best = 0;
#pragma unroll
    for (int k = 0; k < THREADS / WAVE; ++k) {
      const float mk = sh_m[k];
      p.sum += sh_s[k] * (mk == p.max ? 1.0f : exp_from(mk, p.max));
      if (cuts) p.ssum += sh_ss[k] * (mk == p.max ? 1.0f : mk == -INFINITY ? 0.0f : __expf((mk - p.max) * inv_t));
      if (mk == p.max) p.arg = min(p.arg, sh_arg[k]);
      const unsigned long long w = pack_key(sh_key[k], max(sh_tok[k], 0));
      p.best = w > p.best ? w : p.best;
    }
    if (p.arg == 0x7fffffff) p.arg = -1;
    p.edge = INFINITY;
    p.listed = 0;
    p.mass = 0.0f;
  }
  return p;
}

#define SHORT 1024         // tokens that a slice looks at more closely

// The tokens of [lo, hi) near the slice's max M, for a row that truncates: as deep below it as ``cap`` tokens reach, in
// steps of 0.3 of scaled logit (2.5 where a step of that holds more than SHORT), and 20 at most. So with top-k up to
// about cap the cut always lies in the lists: the slice whose list ends first has that many above its end. Two more walks
// over a slice that the caches still hold, by all workgroups at once, for a walk over the whole row by one. False: not
// even the first step fits.
__device__ __forceinline__ bool slice_list(SliceToken* __restrict__ list, int cap, const float* __restrict__ row,
                                           const uint32_t* __restrict__ mrow, float temp, float M, int lo, int hi,
                                           SliceToken* __restrict__ near, float& edge, int& listed, float& mass) {
  constexpr float STEP = 2.5f, FINE = STEP / 8;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float inv_t = (temp > 0.0f) ? 1.0f / temp : 0.0f;
  __shared__ __attribute__((aligned(16))) int counts[8];
  __shared__ int fine[8], put, taken[PT / WAVE];
  __shared__ float red[PT / WAVE];
  if (tid < 8) counts[tid] = fine[tid] = 0;
  if (tid == 8) put = 0;
  __syncthreads();
  auto window = [&](float x) { return (M - x) * inv_t * (1.0f / STEP); };
  auto walk = [&](auto f) {              // f(token, logit, there is one)
    for (int i0 = lo; i0 < hi; i0 += PT * PU) {
      float x[PU];
#pragma unroll
      for (int j = 0; j < PU; ++j) x[j] = row[min(i0 + j * PT + tid, hi - 1)];
#pragma unroll
      for (int j = 0; j < PU; ++j) {
        const int i = i0 + j * PT + tid;
        f(i, x[j], i < hi && (!mrow || ((mrow[i >> 5] >> (i & 31)) & 1)));
      }
    }
  };
  auto plus = [](int p, int q) { return p + q; };
  unsigned long long windows = 0;        // eight counts of 8 bits: a thread has at most 255 tokens
  walk([&](int, float x, bool ok) {
    const float d = window(x);
    if (ok && d < 8.0f) windows += 1ull << (8 * (int)d);
  });
#pragma unroll
  for (int k = 0; k < 4; ++k) {          // two counts of 16 bits a word: 64 lanes fit
    uint32_t w = (uint32_t)(windows >> (16 * k));
    w = (uint32_t)wave_fold((int)((w & 0xff) | (w & 0xff00) << 8), plus);
    if (lane == 0) {
      atomicAdd(&counts[2 * k], (int)(w & 0xffff));
      atomicAdd(&counts[2 * k + 1], (int)(w >> 16));
    }
  }
  __syncthreads();
  int in_window[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) in_window[k] = counts[k];
  int deep = 0, n = 0, next = 0;         // whole windows, their tokens, those of the window behind them
  bool more = true;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    if (more && n + in_window[k] <= cap) n += in_window[k], deep = k + 1;
    else if (more) next = in_window[k], more = false;
  }
  const bool closely = deep < 8 && n + next <= SHORT;
  if (deep == 0 && !closely) return false;
  const int steps = deep + closely;
  // each thread's tokens behind those of the threads before it: their number is in its windows
  int mine = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) mine += k < steps ? (int)(windows >> (8 * k) & 0xff) : 0;
  const int upto = wave_scan(mine);
  if (lane == 63) taken[wave] = upto;
  __syncthreads();
  int at = upto - mine, found = 0;
#pragma unroll
  for (int w = 0; w < PT / WAVE; ++w) {
    at += w < wave ? taken[w] : 0;
    found += taken[w];
  }
  if (found > SHORT) return false;
  walk([&](int i, float x, bool ok) {
    if (ok && window(x) < (float)steps) near[at++] = SliceToken{x, i};
  });
  __syncthreads();
  float from = M - steps * STEP * temp;
  if (closely) {
    for (int e = tid; e < found; e += PT) {
      const float d = (window(near[e].x) - deep) * 8.0f;
      if (d >= 0.0f) atomicAdd(&fine[min((int)d, 7)], 1);
    }
    __syncthreads();
    int k = 0;
    while (k < 8 && n + fine[k] <= cap) n += fine[k++];
    if (deep == 0 && k == 0) return false;
    from = M - (deep * STEP + k * FINE) * temp;
  }
  float sum = 0.0f;
  for (int e0 = 0; e0 < found; e0 += PT) {
    const int e = e0 + tid;
    const SliceToken t = near[min(e, found - 1)];
    const bool in = e < found && t.x >= from;      // a token at a window's end can fall on the other side of ``from``
    const unsigned long long votes = __ballot(in);
    if (!votes) continue;
    int at = 0;
    if (lane == 0) at = atomicAdd(&put, (int)__popcll(votes));
    at = __shfl(at, 0) + (int)__popcll(votes & ((1ull << lane) - 1));
    if (!in) continue;
    sum += __expf((t.x - M) * inv_t);
    if (at < cap) list[at] = t;
  }
  sum = wave_fold(sum, [](float p, float q) { return p + q; });
  if (lane == 0) red[wave] = sum;
  __syncthreads();
  mass = 0.0f;
#pragma unroll
  for (int w = 0; w < PT / WAVE; ++w) mass += red[w];
  listed = put;
  edge = from + (4e-7f * fabsf(M) + 1e-5f * temp);   // above what the windows' rounding can have left out
  return listed <= cap;
}

// Whether a truncated row's slices list their tokens. A top-k that the lists are long enough for lies in them for sure, and
// in a few rows the try is made for one of a quarter more (the top-k 50 of 8 rows of 128256, whose lists hold 48), and for
// what a mask leaves of a row (2 masked rows of 50257, top-p 0.9: 61 us without, 30 with; 16 of 128256: 130 and 118).
// Elsewhere top-p's nucleus is seldom in the lists, and rows whose lists end before their cut pay 3 to 8 % for the try.
__device__ __forceinline__ bool lists_pay(int rows, int V, int top_k, int cap, bool masked) {
  const bool few = (int64_t)rows * V <= 1 << 22;
  return (masked && few) || (top_k > 0 && top_k <= (few ? cap + cap / 4 : cap));
}

// LISTS false: what a call without lists need not carry (its truncated rows are 1 us faster so)
template <bool LISTS>
__global__ void __launch_bounds__(PT) sample_part_kernel(
    SlicePart* __restrict__ parts,        // [B, slices]
    const float* __restrict__ logits,     // [B, V]
    const float* __restrict__ temperatures, const float* __restrict__ top_ps,
    const int* __restrict__ top_ks, const int64_t* __restrict__ seeds,
    const int64_t* __restrict__ steps,
    const uint32_t* __restrict__ mask,    // [B, ceil(V/32)] or nullptr
    SliceToken* __restrict__ lists, int cap,   // [B, slices, cap] or nullptr
    int V, int slice) {
  const int b = blockIdx.y;
  const int lo = blockIdx.x * slice, hi = min(V, lo + slice);
  const float temp = temperatures[b];
  const float* row = logits + (int64_t)b * V;
  const uint32_t* mrow = mask ? mask + (int64_t)b * ((V + 31) / 32) : nullptr;
  const bool cuts = temp != 0.0f && truncates(top_ps[b], top_ks[b], V);
  __shared__ SliceToken room[PT * PU];   // a masked row's allowed tokens, or what slice_list looks at
  static_assert(SHORT <= PT * PU);
  SlicePart p = slice_part<PT>(row, mrow, temp, cuts, draw_base(seeds[b], steps[b]), lo, hi, room);
  const bool pays = LISTS && cuts && lists_pay(gridDim.y, V, top_ks[b], cap, mask != nullptr);
  if (pays) {
    __shared__ float top;
    // without an allowed token there is nothing to list; a max or a sum that is not finite leaves the row to the sweeps
    if (threadIdx.x == 0) top = p.arg < 0 ? -INFINITY : p.sum - p.sum == 0.0f ? p.max : INFINITY;
    __syncthreads();
    float edge = top, mass = 0.0f;
    int listed = 0;
    if (top - top == 0.0f && !slice_list(lists + ((int64_t)b * gridDim.x + blockIdx.x) * cap, cap, row, mrow, temp, top,
                                         lo, hi, room, edge, listed, mass)) {
      edge = INFINITY;
      listed = 0;
      mass = 0.0f;
    }
    p.edge = edge;
    p.listed = listed;
    p.mass = mass;
  }
  if (threadIdx.x == 0) parts[(int64_t)b * gridDim.x + blockIdx.x] = p;
}


// WHOLE: a short row's only launch, one slice of all its tokens
template <bool WHOLE, bool LISTS>
__global__ void __launch_bounds__(NT) sample_final_kernel(
    int64_t* __restrict__ out_tokens,     // [B]
    float* __restrict__ out_logprobs,     // [B]
    const SlicePart* __restrict__ parts,  // [B, slices], slices <= 64
    int slices,
    const SliceToken* __restrict__ lists, int cap,   // [B, slices, cap], slices * cap <= SLIST, or nullptr
    const float* __restrict__ logits,     // [B, V]
    const float* __restrict__ temperatures,
    const float* __restrict__ top_ps,
    const int* __restrict__ top_ks,
    const int64_t* __restrict__ seeds,
    const int64_t* __restrict__ steps,
    const uint32_t* __restrict__ mask,    // [B, ceil(V/32)] or nullptr
    int V, float* __restrict__ dbg) {   // dbg: [B, 16] or nullptr (diagnostics)
  const int b = blockIdx.x;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = tid / WAVE;
  const float* row = logits + (int64_t)b * V;
  const uint32_t* mrow = mask ? mask + (int64_t)b * ((V + 31) / 32) : nullptr;
  const float temp = temperatures[b];
  const float top_p = top_ps[b];
  const int top_k = top_ks[b];
  const float inv_t = (temp > 0.0f) ? 1.0f / temp : 0.0f;
  const bool cuts = temp != 0.0f && truncates(top_p, top_k, V);
  const Draw rng(draw_base(seeds[b], steps[b]), inv_t);

  __shared__ float hist_mass[NW * SBINS];
  __shared__ unsigned int hist_cnt[NW * SBINS];
  auto clear_hist = [&]() {
    for (int i = tid; i < NW * SBINS; i += NT) {
      hist_mass[i] = 0.0f;
      hist_cnt[i] = 0;
    }
  };
  // the lists are on their way before it is known how much of them counts
  SliceToken ahead[SLIST / NT];
  if (LISTS && cuts) {
#pragma unroll
    for (int k = 0; k < SLIST / NT; ++k)
      ahead[k] = lists[(int64_t)b * slices * cap + min(tid + k * NT, slices * cap - 1)];
  }
  __shared__ float sh_max, sh_sum, sh_ssum;
  __shared__ int sh_argmax;
  __shared__ unsigned long long sh_best;
  __shared__ float sh_edge;              // all tokens of the row from this logit on are in the slices' lists
  __shared__ float sh_mass;              // and what those weigh, against the max
  __shared__ int sh_count[64], sh_total;
  if constexpr (WHOLE) {
    const SlicePart p = slice_part<NT>(row, mrow, temp, cuts, draw_base(seeds[b], steps[b]), 0, V, nullptr);
    if (tid == 0) {
      sh_max = p.max;
      sh_sum = p.sum;
      sh_ssum = p.ssum;
      sh_argmax = p.arg < 0 ? 0 : p.arg;
      sh_best = p.best;
    }
  } else if (wid == 0) {
    SlicePart p{-INFINITY, 0.0f, -1, 0.0f, (unsigned long long)NO_KEY << 32, -INFINITY, 0, 0.0f, 0};
    if (lane < slices) p = parts[(int64_t)b * slices + lane];
    auto most = [](float v, float w) { return fmaxf(v, w); };
    auto plus = [](float v, float w) { return v + w; };
    const float M = wave_fold(p.max, most);
    const float S = wave_fold(p.sum * (p.max == M ? 1.0f : exp_from(p.max, M)), plus);
    // a slice without an allowed token has nothing to add
    const float scale = p.max == M ? 1.0f : __expf((p.max - M) * inv_t);
    const float SS = cuts ? wave_fold(p.arg < 0 ? 0.0f : p.ssum * scale, plus) : 0.0f;
    const int a = wave_fold((p.max == M && p.arg >= 0) ? p.arg : 0x7fffffff, [](int v, int w) { return min(v, w); });
    unsigned long long w = 0;
    if (!cuts) w = wave_max_u64(p.best);
    if (LISTS && cuts) {
      const float edge = wave_fold(p.edge, most);
      const float lmass = wave_fold(p.listed == 0 ? 0.0f : p.mass * scale, plus);
      const int total = wave_fold(p.listed, [](int v, int w) { return v + w; });
      sh_count[lane] = p.listed;
      if (lane == 0) {
        sh_edge = edge;
        sh_mass = lmass;
        sh_total = total;
      }
    }
    if (lane == 0) {
      sh_max = M;
      sh_sum = S;
      sh_ssum = SS;
      sh_argmax = a == 0x7fffffff ? 0 : a;
      sh_best = w;
    }
  }
  if (cuts) clear_hist();                // beside the fold
  __syncthreads();
  const float gmax = sh_max;
  const float gsum_unscaled = sh_sum;
  const int argmax_tok = sh_argmax;
  if (!cuts) {
    if (tid == 0) {
      const int tok = (temp == 0.0f || (uint32_t)(sh_best >> 32) == NO_KEY) ? argmax_tok
                                                                           : (int)(sh_best & 0xffffffffu);
      out_tokens[b] = tok;
      out_logprobs[b] = row[tok] - gmax - __logf(gsum_unscaled);
    }
    return;
  }

  __shared__ float list_x[SLIST];
  __shared__ int list_tok[SLIST];
  __shared__ int sh_listed;
  const float smax = gmax * inv_t;
  float* my_mass = hist_mass + wid * SBINS;
  unsigned int* my_cnt = hist_cnt + wid * SBINS;
  // fold the per-wave histograms over bins [from, to): thread j owns bin j; the
  // copy of wave 0 becomes the whole
  auto fold_hist = [&](int from, int to) {
    if (tid >= from && tid < to) {
      float m = 0.0f;
      unsigned int c = 0;
#pragma unroll 4
      for (int w = 0; w < NW; ++w) {
        m += hist_mass[w * SBINS + tid];
        c += hist_cnt[w * SBINS + tid];
      }
      hist_mass[tid] = m;
      hist_cnt[tid] = c;
    }
  };
  // f(token, x, sx) over the row's allowed tokens whose sx is not at or below
  // ``from`` (NaN: all of them). One workgroup hides a sweep's latency by bytes
  // in flight alone: 128 a thread, as 16-byte loads from the row's first aligned
  // token on.
  auto sweep = [&](float from, auto f) {
    auto one = [&](int i, float x) {
      const float sx = sx_of(x, inv_t, smax);
      if (!(sx <= from) && (!mrow || ((mrow[i >> 5] >> (i & 31)) & 1))) f(i, x, sx);
    };
    const int head = min((int)((4 - (((int64_t)b * V) & 3)) & 3), V);
    const int nvec = (V - head) / 4;
    const f32x4* rv = reinterpret_cast<const f32x4*>(row + head);
    for (int i0 = tid; i0 < nvec; i0 += NT * 8) {
      f32x4 x[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = rv[min(i0 + j * NT, nvec - 1)];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int v = i0 + j * NT;
        bool any = false;
#pragma unroll
        for (int k = 0; k < 4; ++k) any |= !(sx_of(x[j][k], inv_t, smax) <= from);
        if (v < nvec && any) {
          const int i = head + v * 4;
          for (int k = 0; k < 4; ++k) one(i + k, k == 0 ? x[j][0] : k == 1 ? x[j][1] : k == 2 ? x[j][2] : x[j][3]);
        }
      }
    }
    if (tid < head) one(tid, row[tid]);
    const int tail = head + nvec * 4 + tid;
    if (tail < V) one(tail, row[tail]);
  };
  auto coarse_bin = [](float sx) { return min((int)(-sx * (SBINS / SRANGE)), SBINS - 1); };

  // boundary-interval state (sx space: 0 at the max, negative below);
  // need_* is the admission still OWED by the boundary interval after
  // everything strictly above it is admitted. MEMBERSHIP in the boundary
  // interval is tested by re-evaluating the PREVIOUS level's exact binning
  // expression (sel_*) — never by interval comparisons, which disagree
  // with the truncating multiply by an ulp at bin edges (and at sx ~ 0).
  __shared__ float sh_lo, sh_hi, sh_need_mass;
  __shared__ float sh_sel_hi, sh_sel_invw;
  __shared__ int sh_sel_cut, sh_sel_coarse, sh_cut;
  __shared__ unsigned int sh_need_cnt;
  __shared__ int sh_state;  // 0 = threshold at sh_lo, 1 = refine, 2 = admit all
  // first of the folded bins [0, n) where the running mass or count meets the
  // need, with what lies before it; -1: none. Wave 0 only, four bins a lane (one
  // thread's walk over 256 bins in LDS takes 14 us)
  auto find_cut = [&](int n, float need_mass, unsigned int need_cnt, float& before_mass, unsigned int& before_cnt) {
    float m[4];
    unsigned int c[4];
    float ms = 0.0f;
    unsigned int cs = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      m[k] = hist_mass[lane * 4 + k];
      c[k] = hist_cnt[lane * 4 + k];
      ms += m[k];
      cs += c[k];
    }
    float mb = wave_before(wave_scan(ms));
    unsigned int cb = wave_before(wave_scan(cs));
    int hit = -1;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (hit < 0) {
        if (lane * 4 + k < n && (mb + m[k] >= need_mass || cb + c[k] >= need_cnt)) {
          hit = lane * 4 + k;
        } else {
          mb += m[k];
          cb += c[k];
        }
      }
    }
    const unsigned long long any = __ballot(hit >= 0);
    if (!any) return -1;
    const int src = __ffsll(any) - 1;
    before_mass = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(mb), src));
    before_cnt = __builtin_amdgcn_readlane(cb, src);
    return __builtin_amdgcn_readlane(hit, src);
  };

  // ---- histogram of the scaled mass, boundary bin --------------------------
  // The bins near the max first, their tokens listed: a peaked row's cut lies
  // there, and the list then stands in for the row.
  // sh_ssum is against the max itself, the bins against smax, its product with 1/T
  // rounded: at a scaled max of 3000 up to 1e-4 apart, which the factor takes out
  const float need_mass = top_p < 1.0f ? top_p * (sh_ssum * __expf(sx_of(gmax, inv_t, smax))) : INFINITY;
  const unsigned int need_cnt = (top_k > 0 && top_k < V) ? (unsigned)top_k : 0xffffffffu;
  // bins that the slices' lists hold whole; their tokens then stand in for the row if the cut lies there
  int whole = 0;
  bool hope = false;
  if constexpr (LISTS) {
    const float deep = -sx_of(sh_edge, inv_t, smax) - 1e-3f;
    whole = deep > 0.0f ? min((int)(deep * (SBINS / SRANGE)), SBINS) : 0;      // NaN: none
    hope = (unsigned)sh_total >= need_cnt || sh_mass * 1.001f >= top_p * sh_ssum;
  }
  if (tid == 0) sh_best = (unsigned long long)NO_KEY << 32;
  // where the cut is behind the lists, the sweeps over bins that those hold whole are left out
  const int after = whole >= SMID ? 2 : whole >= SNEAR ? 1 : 0;
  float best = -INFINITY, best_x = 0.0f;
  int btok = argmax_tok;
  auto consider = [&](int i, float x) {
    const float key = rng.key(i, x);
    if (key > best) { best = key; best_x = x; btok = i; }
  };
  auto finish = [&]() {
    const float K = wave_fold(best, [](float v, float w) { return fmaxf(v, w); });
    const int tok = wave_fold(best == K ? btok : -1, [](int v, int w) { return max(v, w); });
    if (lane == 0) atomicMax(&sh_best, pack_key(K, tok));
    __syncthreads();
    const bool drawn = (uint32_t)(sh_best >> 32) != NO_KEY;
    if (drawn ? pack_key(best, btok) == sh_best : tid == 0) {
      out_tokens[b] = btok;
      out_logprobs[b] = (drawn ? best_x : row[btok]) - gmax - __logf(gsum_unscaled);
    }
  };
  bool fresh = true;                     // the histogram is clear
  int start = whole > 0 && hope ? -1 : after;
  if constexpr (LISTS) {
    // A cut in the lists, and few tokens in its bin: their order is made by one wave, and a thread's tokens stay in
    // registers. Anything else is left to the general way below
    if (start < 0 && !dbg) {
      float sx[SLIST / NT];
      int bin[SLIST / NT];
      if (tid == 0) sh_listed = 0;
#pragma unroll
      for (int k = 0; k < SLIST / NT; ++k) {
        const int e = tid + k * NT;
        sx[k] = sx_of(ahead[k].x, inv_t, smax);
        bin[k] = e < slices * cap && e % cap < sh_count[e / cap] ? coarse_bin(sx[k]) : SBINS;
        if (bin[k] >= whole) bin[k] = SBINS;
        if (bin[k] < SBINS) {
          atomicAdd(&my_mass[bin[k]], __expf(sx[k]));
          atomicAdd(&my_cnt[bin[k]], 1u);
        }
      }
      __syncthreads();
      fold_hist(0, whole);
      __syncthreads();
      if (wid == 0) {
        float before_mass = 0.0f;
        unsigned int before_cnt = 0;
        const int cut_bin = find_cut(whole, need_mass, need_cnt, before_mass, before_cnt);
        if (lane == 0) {
          sh_cut = cut_bin;
          sh_need_mass = need_mass - before_mass;
          sh_need_cnt = need_cnt == 0xffffffffu ? need_cnt : need_cnt - before_cnt;
        }
      }
      __syncthreads();
      const int cut = sh_cut;
      const unsigned int n = cut < 0 ? 0 : hist_cnt[cut];
      // with no mass left to fill (top-p 0) what ties with the max is in, which the general way finds
      if (cut >= 0 && n <= WAVE && sh_need_mass > 0.0f) {
#pragma unroll
        for (int k = 0; k < SLIST / NT; ++k)
          if (bin[k] == cut) {
            const int at = atomicAdd(&sh_listed, 1);
            list_x[at] = ahead[k].x;
            list_tok[at] = ahead[k].tok;
          }
#pragma unroll
        for (int k = 0; k < SLIST / NT; ++k)
          if (bin[k] < cut) consider(ahead[k].tok, ahead[k].x);
        __syncthreads();
        if (wid == 0) {
          // what of the bin lies above a token; equal ones are in or out together, as in the general way
          const float x = list_x[lane < (int)n ? lane : 0], s = sx_of(x, inv_t, smax), e = __expf(s);
          float above = 0.0f;
          unsigned int higher = 0;
          for (unsigned int j = 0; j < n; ++j) {
            const bool over = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(s), j)) > s;
            above += over ? __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(e), j)) : 0.0f;
            higher += over;
          }
          if (lane < (int)n && above < sh_need_mass && higher < sh_need_cnt) consider(list_tok[lane], x);
        }
        finish();
        return;
      }
      fresh = false;
      if (cut < 0) start = after;
    }
  }
  bool listing = false;                  // whether the part that found the cut, with those it adds to, listed its tokens
  for (int part = start; part < 3; part = part < 0 ? after : part + 1) {
    const int from = part <= after ? 0 : part == 1 ? SNEAR : SMID;
    const int to = part < 0 ? whole : part == 0 ? SNEAR : part == 1 ? SMID : SBINS;
    listing = part < 2;
    if (part <= after) {
      if (!fresh) {
        __syncthreads();
        clear_hist();
      }
      fresh = false;
      if (tid == 0) sh_listed = 0;
      __syncthreads();
    }
    auto count = [&](int i, float x, float sx, int bin) {
      atomicAdd(&my_mass[bin], __expf(sx));
      atomicAdd(&my_cnt[bin], 1u);
      if (listing) {
        const int at = atomicAdd(&sh_listed, 1);
        if (at < SLIST) {
          list_x[at] = x;
          list_tok[at] = i;
        }
      }
    };
    if (part < 0) {
#pragma unroll
      for (int k = 0; k < SLIST / NT; ++k) {
        const int e = tid + k * NT;
        if (e >= slices * cap || e % cap >= sh_count[e / cap]) continue;
        const float sx = sx_of(ahead[k].x, inv_t, smax);
        const int bin = coarse_bin(sx);
        if (bin < to) count(ahead[k].tok, ahead[k].x, sx, bin);
      }
    } else {
      sweep(part < 2 ? -to * (SRANGE / SBINS) - 1e-3f : NAN, [&](int i, float x, float sx) {
        const int bin = coarse_bin(sx);
        if (bin >= from && bin < to) count(i, x, sx, bin);
      });
    }
    __syncthreads();
    fold_hist(from, to);
    __syncthreads();
    if (wid == 0) {
      float before_mass = 0.0f;
      unsigned int before_cnt = 0;
      const int cut_bin = find_cut(to, need_mass, need_cnt, before_mass, before_cnt);
      if (lane == 0) {
        if (cut_bin < 0) {
          sh_state = 2;  // window never met the need: admit everything
          sh_cut = SBINS;
          sh_lo = -INFINITY;
        } else {
          const float binw = SRANGE / SBINS;
          sh_lo = -(cut_bin + 1) * binw;
          sh_hi = -cut_bin * binw;
          sh_need_mass = need_mass - before_mass;
          sh_need_cnt = (need_cnt == 0xffffffffu) ? 0xffffffffu : need_cnt - before_cnt;
          sh_sel_coarse = 1;
          sh_sel_cut = cut_bin;
          sh_cut = cut_bin;
          // the whole bin is exactly owed -> no refinement needed
          sh_state = (hist_cnt[cut_bin] == sh_need_cnt) ? 0 : 1;
          if (dbg) {
            dbg[b * 16 + 0] = (float)cut_bin;
            dbg[b * 16 + 1] = (float)hist_cnt[cut_bin];
            dbg[b * 16 + 2] = (float)sh_need_cnt;
            dbg[b * 16 + 3] = (float)sh_state;
          }
        }
      }
    }
    __syncthreads();
    if (sh_cut < SBINS) {
      if (part >= 0) whole = 0;
      break;
    }
  }

  // ---- draw over the bins above the boundary --------------------------------
  // afterwards the list holds the boundary bin's tokens, among others, unless
  // they outgrow it. Part 2 lists nothing, and behind the slices' lists it may
  // end in any bin: their tokens added up in another order can reach a top-p that
  // the lists' sum missed by its rounding
  const int cut = sh_cut;
  const bool near = listing && (cut < SMID || cut < whole) && sh_listed <= SLIST;   // whole: of the lists that were used, else 0
  const bool fits = near || (cut < SBINS && hist_cnt[cut] <= SLIST);
  if (near) {
    const int n = sh_listed;
    for (int e = tid; e < n; e += NT)
      if (coarse_bin(sx_of(list_x[e], inv_t, smax)) < cut) consider(list_tok[e], list_x[e]);
  } else {
    __syncthreads();
    if (tid == 0) sh_listed = 0;
    __syncthreads();
    sweep(cut == SBINS ? NAN : -(cut + 1) * (SRANGE / SBINS) - 1e-3f, [&](int i, float x, float sx) {
      const int bin = coarse_bin(sx);
      if (cut == SBINS || bin < cut) {
        consider(i, x);
      } else if (fits && bin == cut) {
        const int at = atomicAdd(&sh_listed, 1);
        if (at < SLIST) {
          list_x[at] = x;
          list_tok[at] = i;
        }
      }
    });
  }
  __syncthreads();
  const int listed = min(sh_listed, SLIST);
  // f(token, x, sx) over the boundary bin's tokens
  auto boundary = [&](auto f) {
    if (fits) {
      for (int e = tid; e < listed; e += NT) {
        const float x = list_x[e], sx = sx_of(x, inv_t, smax);
        if (coarse_bin(sx) == cut) f(list_tok[e], x, sx);
      }
    } else {
      sweep(NAN, [&](int i, float x, float sx) {
        if (coarse_bin(sx) == cut) f(i, x, sx);
      });
    }
  };

  // refinement: re-histogram ONLY the boundary interval at 256x finer
  // resolution; each level divides the threshold uncertainty by SBINS
  for (int it = 0; it < 3; ++it) {
    if (sh_state != 1) break;
    const float lo = sh_lo, hi = sh_hi;
    const float inv_w = SBINS / (hi - lo);
    const int sel_coarse = sh_sel_coarse;
    const int sel_cut = sh_sel_cut;
    const float sel_hi = sh_sel_hi;
    const float sel_invw = sh_sel_invw;
    clear_hist();
    __syncthreads();
    boundary([&](int, float, float sx) {
      // membership = the EXACT bin the previous level counted this token
      // into equals its boundary bin (bit-identical re-evaluation)
      if (!sel_coarse && min(max((int)((sel_hi - sx) * sel_invw), 0), SBINS - 1) != sel_cut) return;
      int bn = (int)((hi - sx) * inv_w);
      bn = min(max(bn, 0), SBINS - 1);
      atomicAdd(&my_mass[bn], __expf(sx));
      atomicAdd(&my_cnt[bn], 1u);
    });
    __syncthreads();
    fold_hist(0, SBINS);
    __syncthreads();
    if (wid == 0) {
      float before_mass = 0.0f;
      unsigned int before_cnt = 0;
      int cut_bin = find_cut(SBINS, sh_need_mass, sh_need_cnt, before_mass, before_cnt);
      if (cut_bin < 0) {
        // the need is met inside [lo, hi) up to the rounding of the sums: the
        // last bin, with all the others before it
        cut_bin = SBINS - 1;
        before_mass = 0.0f;
        before_cnt = 0;
        for (int k = 0; k < 4; ++k) {
          const int bn = lane * 4 + k;
          before_mass += bn < SBINS - 1 ? hist_mass[bn] : 0.0f;
          before_cnt += bn < SBINS - 1 ? hist_cnt[bn] : 0u;
        }
        before_mass = wave_fold(before_mass, [](float v, float w) { return v + w; });
        before_cnt = wave_fold(before_cnt, [](unsigned int v, unsigned int w) { return v + w; });
      }
      if (lane == 0) {
        const float subw = (hi - lo) / SBINS;
        sh_need_mass -= before_mass;
        if (sh_need_cnt != 0xffffffffu) sh_need_cnt -= before_cnt;
        sh_lo = hi - (cut_bin + 1) * subw;
        sh_hi = hi - cut_bin * subw;
        sh_sel_coarse = 0;
        sh_sel_cut = cut_bin;
        sh_sel_hi = hi;
        sh_sel_invw = inv_w;
        sh_state = (hist_cnt[cut_bin] == sh_need_cnt) ? 0 : 1;
        if (dbg) {
          dbg[b * 16 + 4 + it * 4 + 0] = (float)cut_bin;
          dbg[b * 16 + 4 + it * 4 + 1] = (float)hist_cnt[cut_bin];
          dbg[b * 16 + 4 + it * 4 + 2] = (float)sh_need_cnt;
          dbg[b * 16 + 4 + it * 4 + 3] = sh_lo;
          if (it == 0) {
            dbg[b * 16 + 12] = (float)hist_cnt[0];
            dbg[b * 16 + 13] = sx_of(row[argmax_tok], inv_t, smax);
            dbg[b * 16 + 14] = smax;
            dbg[b * 16 + 15] = __fmul_rn(row[argmax_tok], inv_t);
          }
        }
      }
    }
    __syncthreads();
  }

  // ---- draw over what the boundary bin admits ------------------------------
  if (cut < SBINS) {
    // the threshold stays in sx space (converting it back to x loses the
    // refined margin to fp32 rounding), exclusive at its lower edge as the bins
    const float thresh = sh_lo;
    boundary([&](int i, float x, float sx) {
      if (sx > thresh) consider(i, x);
    });
  }
  finish();
}

// rows -> slices: at most eight 256-thread workgroups per compute unit, which are there at once (120 rows in 18 slices were
// 2160, whose last ones ran alone), and whole load rounds of 2048 tokens as far as may be; at most 64 slices a row (one
// per lane of sample_final's fold). 0: rows of up to 4096 tokens, half a load round of
// sample_final's workgroup, take its launch alone: called from Python 9.0 us against 12.5
// for any number of rows of 300 to 4000 tokens, in a graph 6 to 8 against 8 to 9.5
extern "C" int sample_slices(int B, int V) {
  if (V <= 4 * NT) return 0;
  const int most = (V + PT * PU - 1) / (PT * PU);
  const int want = 2048 / B;
  int n = want < most ? want : most;
  n = n < 1 ? 1 : n > 64 ? 64 : n;
  if ((int64_t)B * n < 1024) return n;   // compute units are left over
  const int rounds = (V + n * PT * PU - 1) / (n * PT * PU);
  return (V + rounds * PT * PU - 1) / (rounds * PT * PU);
}

// Tokens of a slice's list, or 0: no lists. They cost two more walks over the truncated rows by all workgroups and save the
// walks of sample_final, one workgroup a row, so they pay on all but the smallest calls, up to the rows at which
// sample_final's workgroups fill the chip by themselves. us without lists and with, top-p 0.95 and top-k 50, all rows truncated,
// masked with one in eight allowed in brackets:
//   1 row of 32000 14.6, 17.8 (13.6, 18.6)   50257 14.0, 16.9 (30.9, 19.1)   128256 19.4, 16.6 (30.9, 18.1)   8 rows of 8192 18.9, 18.5
//   (18.9, 16.7)   40 of 32000 28.4, 20.1 (27.1, 21.4)   120 of 50257 39.1, 31.0 (40.9, 34.1)   250 of 32000 37.7, 33.1 (37.8,
//   38.6)   250 of 152064 102.7, 83.0 (121.1, 105.4)   512 of 50257 85.3, 69.0 (88.0, 88.0)   1024 of 32000 103.9, 121.4 (107.6, 160.7)
// and half of the rows truncated: 120 of 32000 31.9, 22.7 (31.4, 23.0)   512 of 50257 67.0, 53.0 (63.3, 68.2). Nor have slices
// lists whose threads would count more than 255 tokens.
static int sample_cap(int B, int V, int n, bool masked) {
  return n > 0 && B <= (masked ? 256 : 512) && (int64_t)B * V >= (masked ? 50000 : 120000) && (V + n - 1) / n <= 255 * PT ? SLIST / n : 0;
}

// words of 8 bytes that a call needs for its slices, and for their lists
extern "C" int64_t sample_room(int B, int V, int masked) {
  const int n = sample_slices(B, V);
  return (int64_t)B * n * (sizeof(SlicePart) / 8 + sample_cap(B, V, n, masked));
}

extern "C" void launch_sample(int64_t* tokens, float* logprobs, void* parts, const float* logits,
                              const float* temps, const float* top_ps, const int* top_ks,
                              const int64_t* seeds, const int64_t* steps, const uint32_t* mask, int B,
                              int V, float* dbg, hipStream_t stream) {
  const int n = sample_slices(B, V);
  const int slice = n > 0 ? ((V + n - 1) / n + 63) / 64 * 64 : V;    // whole words of the masks
  const int cap = sample_cap(B, V, n, mask != nullptr);
  SliceToken* lists = cap ? (SliceToken*)((SlicePart*)parts + (int64_t)B * n) : nullptr;   // B is one launch's
  // rows of a launch lie on the grid's y, which ends at 65535
  for (int b = 0; b < B; b += 65535) {
    const int rows = B - b < 65535 ? B - b : 65535;
    SlicePart* p = (SlicePart*)parts + (int64_t)b * n;
    const float* x = logits + (int64_t)b * V;
    const uint32_t* m = mask ? mask + (int64_t)b * ((V + 31) / 32) : nullptr;
    if (n > 0)
      hipLaunchKernelGGL(lists ? sample_part_kernel<true> : sample_part_kernel<false>, dim3(n, rows), dim3(PT), 0, stream, p, x,
                         temps + b, top_ps + b, top_ks + b, seeds + b, steps + b, m, lists, cap, V, slice);
    hipLaunchKernelGGL((n == 0 ? sample_final_kernel<true, false> : lists ? sample_final_kernel<false, true> : sample_final_kernel<false, false>),
                       dim3(rows), dim3(NT), 0, stream,
                       tokens + b, logprobs + b, (const SlicePart*)p, n, (const SliceToken*)lists, cap, x, temps + b, top_ps + b, top_ks + b,
                       seeds + b, steps + b, m, V, dbg ? dbg + (int64_t)b * 16 : nullptr);
  }
}
