// Whole sublayers of a hybrid model's decode step (one row a sequence, up to 128 of them), launched from here one
// kernel behind the other. A step is some 50 launches of 4 to 18 us, and from Python a launch costs the host 12 to 15 us:
// it was the bound (85 launches for 40 rows of the 2048-wide preset: 1310 us, the kernels 775). Here it is 2 to 3.

#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <hip/hip_bf16.h>

#include <algorithm>
#include <optional>

extern "C" {
void seq_launch_sandwich_rows(float*, const float*, int, const float*, int, const float*, const float*, const float*,
                              const float*, void*, int, int, float, const float*, int, float, hipStream_t);
bool seq_parallel_rows_takes(int, int);
void seq_launch_parallel_rows(const float*, int, const void*, const int64_t*, const int64_t*, const float*, void*, void*,
                              const int64_t*, void*, void*, const float*, float*, const float*, void*, float*, const int*,
                              const int*, const int*, int, int, int, int, int, int, int, int, int, hipStream_t);
void seq_launch_gated_rmsnorm(void*, const float*, const float*, const void*, int, int, int, int, float, int,
                              int, hipStream_t);
void seq_launch_causal_conv_silu(void*, const void*, const float*, void*, const int*, const int*, const int*,
                                 const int*, const float*, int, int, int, int, int, int, hipStream_t);
void seq_launch_gated_delta_rule(float*, const void*, const void*, const void*, const void*, const void*,
                                 const float*, const float*, float*, float*, float*, float*, float*, float*,
                                 const int*, const int*, const int*, int, int, int, int, int, int, int, int, int,
                                 int, int, int, float*, hipStream_t);
bool seq_delta_rows_takes(int, int, int, int, int, int, int);
void seq_launch_delta_rows(const float*, int, const int64_t*, const float*, void*, int, int, const void*, int, const void*, int,
                           const float*, const float*, float*, const float*, void*, const int*, const int*, const int*, int,
                           int, int, int, int, int, float, hipStream_t);
void seq_launch_gated_act(void*, const void*, const void*, int64_t, int, int, float, float, float, int, hipStream_t);
// few-row products and paged decode attention (ops/hip/linear_rows.hip, attn_decode.hip, also part of kllms_amd._C)
int launch_linear_rows(void*, const __hip_bfloat16*, const __hip_bfloat16*, const __hip_bfloat16*, int, int, int, int,
                        int, int, float, float, bool, hipStream_t);
int launch_linear_rows_two(float*, const __hip_bfloat16*, const __hip_bfloat16*, const __hip_bfloat16*, int, int, int, int,
                           bool, hipStream_t);
int linear_rows_splits(int, int, int);
int attn_decode_splits(int, int, int, int, int, int, int);
void launch_attn_decode(__hip_bfloat16*, float*, int*, int, const __hip_bfloat16*, const void*, const void*, const float*,
                        const float*, const int*, const int*, const __hip_bfloat16*, int, float, int, int, int, int, int,
                        int, int, int, int, hipStream_t);
}

using torch::Tensor;

namespace {

enum { ROWS_PART = 0, ROWS_BF16 = 1, ROWS_CLAMPED = 4 };   // forms of linear_rows
constexpr const char* NO_LDS = "160 KB of LDS are not available";

inline hipStream_t cur_stream() { return at::hip::getCurrentHIPStream().stream(); }

inline void check(const Tensor& t, at::ScalarType type, int64_t numel, const char* name) {
  TORCH_CHECK(t.is_cuda() && t.scalar_type() == type && t.is_contiguous() && t.numel() == numel, name,
              ": a contiguous GPU tensor of ", numel, " ", toString(type), " values");
}
inline void on_16(const Tensor& t, const char* name) {
  TORCH_CHECK(reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0, name, " must begin on 16 bytes");
}
inline const __hip_bfloat16* bf(const Tensor& t) { return (const __hip_bfloat16*)t.data_ptr(); }
inline const __hip_bfloat16* bf(const Tensor& t, int64_t col) { return bf(t) + col; }

// How the kernels here read weights: contiguous and from 16 bytes on. Others are the general sublayers'
bool lie_whole(std::initializer_list<Tensor> ws) {
  for (const Tensor& w : ws)
    if (!w.is_contiguous() || reinterpret_cast<uintptr_t>(w.data_ptr()) % 16) return false;
  return true;
}

void check_weight(const Tensor& w, int64_t K, const char* name) {
  TORCH_CHECK(w.dim() == 2 && w.size(1) == K && K % 128 == 0 && w.size(0) % 16 == 0, name, ": [N, K], N % 16, K % 128");
  check(w, at::kBFloat16, w.numel(), name);
}

// x [T, K] (contiguous) by w: fp32 sums [S, T, N]
Tensor part(const Tensor& x, const Tensor& w, int T, bool once, hipStream_t st) {
  const int K = w.size(1), N = w.size(0), S = linear_rows_splits(T, N, K);
  auto out = torch::empty({S, T, N}, x.options().dtype(torch::kFloat));
  TORCH_CHECK(launch_linear_rows(out.data_ptr(), bf(x), bf(w), nullptr, T, N, K, K, ROWS_PART, S, 0.0f, 0.0f, once, st) == 0, NO_LDS);
  return out;
}

struct Rows {
  int T, W;
  Rows(const Tensor& x, const Tensor& h) : T(h.size(0)), W(h.size(1)) {
    TORCH_CHECK(h.dim() == 2 && T >= 1 && T <= 128 && W % 128 == 0 && W <= 8192, "1 to 128 rows of a width % 128, <= 8192");
    check(h, at::kBFloat16, (int64_t)T * W, "h");
    check(x, at::kFloat, (int64_t)T * W, "x");
    on_16(h, "h");
    on_16(x, "x");
  }
  void norm(const Tensor& w, const char* name) const { check(w, at::kFloat, W, name); }
};

}  // namespace

// x (fp32 stream, in place) through a parallel sublayer; h = its normed input. y columns: o_lq, o_lk of the softmax
// branch's q and k, o_lg of its head gates; o_rq, o_rk, o_rv, o_rg of the recurrent branch. Returns the next normed input,
// or nothing where the weights lie otherwise than the kernels read them: then nothing has been done
std::optional<Tensor> hybrid_parallel_rows(Tensor x, Tensor h, Tensor w_in, Tensor bias, std::vector<int64_t> at, Tensor inv_freq,
                            Tensor k_cache, Tensor v_cache, Tensor o_left, Tensor decay, Tensor state, Tensor norm_right,
                            Tensor o_right, Tensor wa, Tensor wb, Tensor w_post, Tensor w_next, Tensor positions,
                            Tensor slots, Tensor tables, Tensor lens, Tensor state_slots, Tensor cu, Tensor seg_start,
                            int64_t heads, double scale, int64_t mask_size, double eps, bool once) {
  if (!lie_whole({w_in, o_left, o_right, state, wa, wb, w_post, w_next})) return std::nullopt;
  const Rows r(x, h);
  const int T = r.T, W = r.W;
  check_weight(w_in, W, "w_in");
  const int N = w_in.size(0);
  if (bias.numel()) check(bias, at::kBFloat16, N, "bias");
  TORCH_CHECK(k_cache.dim() == 4 && v_cache.sizes() == k_cache.sizes() && k_cache.size(3) == 128, "caches [NB, G, BS, 128]");
  check(k_cache, at::kBFloat16, k_cache.numel(), "k_cache");
  check(v_cache, at::kBFloat16, k_cache.numel(), "v_cache");
  const int H = heads, G = k_cache.size(1), BS = k_cache.size(2), D = 128;
  TORCH_CHECK(H % G == 0 && (H / G == 1 || H / G == 2 || H / G == 4 || H / G == 8), "heads to a kv head: 1, 2, 4 or 8");
  TORCH_CHECK((int64_t)k_cache.size(0) * G * BS < (1LL << 31) && mask_size >= 0);
  TORCH_CHECK(state.dim() == 4, "state [slots, H, D, V]");
  const int RH = state.size(1), RD = state.size(2), RV = state.size(3);
  check(state, at::kFloat, state.numel(), "state");
  check(decay, at::kFloat, RH, "decay");
  check(norm_right, at::kFloat, (int64_t)RH * RV, "norm_right");
  TORCH_CHECK(RD <= 256 && RD % 4 == 0 && RV % 4 == 0, "key sizes of the recurrence kernel: up to 256, in fours");
  check_weight(o_left, (int64_t)H * D, "o_left");
  check_weight(o_right, (int64_t)RH * RV, "o_right");
  TORCH_CHECK(o_left.size(0) == W && o_right.size(0) == W);
  const int64_t sizes[7] = {(int64_t)H * D, (int64_t)G * D, H, (int64_t)RH * RD, (int64_t)RH * RD, (int64_t)RH * RV,
                            (int64_t)RH * RV};
  TORCH_CHECK(at.size() == 7, "seven column ranges");
  for (int i = 0; i < 7; ++i) TORCH_CHECK(at[i] >= 0 && at[i] % 8 == 0 && at[i] + sizes[i] <= N, "columns of w_in");
  r.norm(wa, "wa"); r.norm(wb, "wb"); r.norm(w_post, "w_post"); r.norm(w_next, "w_next");
  const int R = inv_freq.numel();
  check(inv_freq, at::kFloat, R, "inv_freq");
  TORCH_CHECK(2 * R <= D, "rotary width exceeds the head size");
  check(positions, at::kLong, T, "positions");
  check(slots, at::kLong, T, "slots");
  check(lens, at::kInt, T, "lens");
  check(state_slots, at::kInt, T, "state_slots");
  check(cu, at::kInt, T + 1, "cu");
  check(seg_start, at::kInt, T, "seg_start");
  TORCH_CHECK(tables.dim() == 2 && tables.size(0) == T, "one table row for each row");
  check(tables, at::kInt, tables.numel(), "tables");
  const int width = tables.size(1);
  if (!seq_parallel_rows_takes(RD, RV)) return std::nullopt;

  auto st = cur_stream();
  const auto f32 = x.options();
  const Tensor y = part(h, w_in, T, once, st);
  const int KL = H * D, KR = RH * RV;
  auto q = torch::empty({T, (int64_t)KL}, h.options()), head_gate = torch::empty({T, H}, h.options());
  auto both = torch::empty({(int64_t)T * (KL + KR)}, h.options());     // the left branch's rows, then the right one's
  auto squares = torch::empty({T, RH}, f32);
  seq_launch_parallel_rows(y.data_ptr<float>(), y.size(0), bias.numel() ? bias.data_ptr() : nullptr, at.data(),
                           positions.data_ptr<int64_t>(), inv_freq.data_ptr<float>(), k_cache.data_ptr(), v_cache.data_ptr(),
                           slots.data_ptr<int64_t>(), q.data_ptr(), head_gate.data_ptr(), decay.data_ptr<float>(),
                           state.data_ptr<float>(), norm_right.data_ptr<float>(),
                           (void*)bf(both, (int64_t)T * KL), squares.data_ptr<float>(), state_slots.data_ptr<int>(),
                           cu.data_ptr<int>(), seg_start.data_ptr<int>(), T, N, H, G, R, BS, RH, RD, RV, st);
  const int64_t longest = mask_size > 0 ? std::min<int64_t>(mask_size, (int64_t)width * BS) : (int64_t)width * BS;
  const int longest32 = (int)std::min<int64_t>(longest, INT32_MAX);
  const int splits = attn_decode_splits(T, G, H / G, longest32, 0, 1, 0);
  auto partials = torch::empty({splits > 1 ? (int64_t)T * H * splits * 130 : 0}, f32);
  launch_attn_decode((__hip_bfloat16*)both.data_ptr(), partials.data_ptr<float>(), nullptr, 1, bf(q), k_cache.data_ptr(),
                     v_cache.data_ptr(), nullptr, nullptr, tables.data_ptr<int>(), lens.data_ptr<int>(), bf(head_gate), H,
                     (float)scale, H, G, BS, width, longest32, KL, T, 0, (int)mask_size, st);
  Tensor left, right;
  if (KL == KR) {    // one launch, half as many sums of each: 40 rows, 2048 x 2048 each, 6.2 us, two launches 5.3 each
    const int S = std::max(linear_rows_splits(T, W, 2 * KL) & ~1, 2);
    const Tensor sums = torch::empty({S, T, (int64_t)W}, f32);
    TORCH_CHECK(launch_linear_rows_two(sums.data_ptr<float>(), bf(both), bf(o_left), bf(o_right), T, W, KL, S, once, st) == 0, NO_LDS);
    left = sums.narrow(0, 0, S / 2);
    right = sums.narrow(0, S / 2, S / 2);
  } else {
    left = part(both, o_left, T, once, st);
    right = part(both.narrow(0, (int64_t)T * KL, (int64_t)T * KR), o_right, T, once, st);
  }
  auto out = torch::empty_like(h);
  seq_launch_sandwich_rows(x.data_ptr<float>(), left.data_ptr<float>(), left.size(0), right.data_ptr<float>(),
                           right.size(0), wa.data_ptr<float>(), wb.data_ptr<float>(), w_post.data_ptr<float>(),
                           w_next.data_ptr<float>(), out.data_ptr(), T, W, (float)eps, squares.data_ptr<float>(), RH,
                           1.0f / (float)KR, st);
  return out;
}

// The same of a gated-delta-rule sublayer. at: columns of q, k, v, of the two low-rank inputs and of the write strengths
std::optional<Tensor> hybrid_delta_rows(Tensor x, Tensor h, Tensor w_in, std::vector<int64_t> at, Tensor conv, Tensor conv_state, Tensor a2,
                         Tensor g2, Tensor dt_bias, Tensor a_log, Tensor state, Tensor norm, Tensor w_out, Tensor w_post,
                         Tensor w_next, Tensor state_slots, Tensor cu, Tensor seg_start, Tensor token_seg,
                         int64_t kv_heads, double eps, bool once) {
  if (!lie_whole({w_in, w_out, w_post, w_next})) return std::nullopt;
  const Rows r(x, h);
  const int T = r.T, W = r.W;
  check_weight(w_in, W, "w_in");
  const int N = w_in.size(0);
  TORCH_CHECK(state.dim() == 4, "state [slots, H, D, V]");
  const int H = state.size(1), D = state.size(2), V = state.size(3), G = kv_heads;
  check(state, at::kFloat, state.numel(), "state");
  TORCH_CHECK(G >= 1 && H % G == 0 && D <= 256, "heads and key size of the recurrence");
  TORCH_CHECK(a2.dim() == 2 && g2.dim() == 2 && a2.size(0) == (int64_t)H * D && g2.size(0) == (int64_t)H * V);
  const int64_t sizes[6] = {(int64_t)G * D, (int64_t)G * D, (int64_t)H * V, a2.size(1), g2.size(1), H};
  TORCH_CHECK(at.size() == 6, "six column ranges");
  for (int i = 0; i < 6; ++i) TORCH_CHECK(at[i] >= 0 && at[i] % 8 == 0 && at[i] + sizes[i] <= N, "columns of w_in");
  TORCH_CHECK(conv.dim() == 2 && conv_state.dim() == 3, "taps [K, C], history [slots, K - 1, C]");
  const int K = conv.size(0), C = conv.size(1);
  for (int i = 0; i < 3; ++i) TORCH_CHECK(at[i] + sizes[i] <= C && C <= N, "the convolution's columns");
  check(conv, at::kFloat, (int64_t)K * C, "conv");
  check(conv_state, at::kBFloat16, conv_state.numel(), "conv_state");
  TORCH_CHECK(K >= 1 && K <= 16 && conv_state.size(1) == K - 1 && conv_state.size(2) == C);
  check(dt_bias, at::kFloat, (int64_t)H * D, "dt_bias");
  check(a_log, at::kFloat, H, "a_log");
  check(norm, at::kFloat, V, "norm");
  check_weight(w_out, (int64_t)H * V, "w_out");
  TORCH_CHECK(w_out.size(0) == W);
  r.norm(w_post, "w_post"); r.norm(w_next, "w_next");
  check(state_slots, at::kInt, T, "state_slots");
  check(cu, at::kInt, T + 1, "cu");
  check(seg_start, at::kInt, T, "seg_start");
  check(token_seg, at::kInt, T, "token_seg");

  auto st = cur_stream();
  auto yr = torch::empty({T, (int64_t)H * V}, h.options());
  if (lie_whole({a2, g2, state}) && a2.scalar_type() == at::kBFloat16 && g2.scalar_type() == at::kBFloat16 &&
      seq_delta_rows_takes(H, G, D, V, K, a2.size(1), g2.size(1))) {
    const Tensor y = part(h, w_in, T, once, st);
    seq_launch_delta_rows(y.data_ptr<float>(), y.size(0), at.data(), conv.data_ptr<float>(), conv_state.data_ptr(), K, C,
                          a2.data_ptr(), a2.size(1), g2.data_ptr(), g2.size(1), dt_bias.data_ptr<float>(),
                          a_log.data_ptr<float>(), state.data_ptr<float>(), norm.data_ptr<float>(), yr.data_ptr(),
                          state_slots.data_ptr<int>(), cu.data_ptr<int>(), seg_start.data_ptr<int>(), T, N, H, G, D, V,
                          (float)eps, st);
  } else {
    // the kernels of the general sublayer, launched from here: a step of 8 rows of the 2048-wide preset with ranks of 60 648 us
    // with them from Python, 499 so
    const auto f32 = x.options();
    auto y = torch::empty({T, (int64_t)N}, h.options());
    TORCH_CHECK(launch_linear_rows(y.data_ptr(), bf(h), bf(w_in), nullptr, T, N, W, W, ROWS_BF16, 1, 0.0f, 0.0f, once, st) == 0, NO_LDS);
    auto c = torch::empty({T, C}, h.options());
    seq_launch_causal_conv_silu(c.data_ptr(), y.data_ptr(), conv.data_ptr<float>(), conv_state.data_ptr(),
                                state_slots.data_ptr<int>(), cu.data_ptr<int>(), seg_start.data_ptr<int>(),
                                token_seg.data_ptr<int>(), nullptr, T, T, C, K, N, 0, st);
    const Tensor a = at::linear(y.narrow(1, at[3], sizes[3]), a2), gate = at::linear(y.narrow(1, at[4], sizes[4]), g2);
    auto o = torch::empty({T, (int64_t)H * V}, f32), qn = torch::empty({T, (int64_t)G * D}, f32),
         kn = torch::empty({T, (int64_t)G * D}, f32), gd = torch::empty({T, (int64_t)H * D}, f32),
         vf = torch::empty({T, (int64_t)H * V}, f32), bt = torch::empty({T, H}, f32);
    seq_launch_gated_delta_rule(o.data_ptr<float>(), bf(c, at[0]), bf(c, at[1]), bf(c, at[2]), bf(y, at[5]), a.data_ptr(),
                                dt_bias.data_ptr<float>(), a_log.data_ptr<float>(), qn.data_ptr<float>(),
                                kn.data_ptr<float>(), gd.data_ptr<float>(), vf.data_ptr<float>(), bt.data_ptr<float>(),
                                state.data_ptr<float>(), state_slots.data_ptr<int>(), cu.data_ptr<int>(),
                                seg_start.data_ptr<int>(), T, T, H, G, D, V, C, C, C, N, H * D, 0, nullptr, st);
    seq_launch_gated_rmsnorm(yr.data_ptr(), o.data_ptr<float>(), norm.data_ptr<float>(), gate.data_ptr(), T, H, V, H * V,
                             (float)eps, 0, 0, st);
  }
  const Tensor p = part(yr, w_out, T, once, st);
  auto out = torch::empty_like(h);
  seq_launch_sandwich_rows(x.data_ptr<float>(), p.data_ptr<float>(), p.size(0), nullptr, 0, nullptr, nullptr,
                           w_post.data_ptr<float>(), w_next.data_ptr<float>(), out.data_ptr(), T, W, (float)eps, nullptr, 0, 0.0f, st);
  return out;
}

// Whether the gated product of T rows is the few-row kernel's, which has the activation in it, or the library's and a pass
// behind it. us of the one and the other by T, w_in of 16384 x 2048: 1 13.8, 19.6   64 15.2, 20.6   128 18.8, 23.6; 28672 x 4096: 16
// 41.6, 62.8   128 50.9, 57.5; 57344 x 8192: 16 166, 186   128 197, 203; of other widths than powers of two the stages take a
// third longer at many rows: 27648 x 5120 16 57, 82   64 62, 60   128 85, 70; 24576 x 3072 96 41, 39   128 49, 43
static bool glu_on_rows(int T, int K) { return T <= 64 || (K & (K - 1)) == 0; }

// The same of a clamped gated-linear-unit sublayer, w_in = [gate; up]
std::optional<Tensor> hybrid_glu_rows(Tensor x, Tensor h, Tensor w_in, Tensor w_down, Tensor w_post, Tensor w_next, double limit,
                       double alpha, double eps, bool once) {
  if (!lie_whole({w_in, w_down, w_post, w_next})) return std::nullopt;
  const Rows r(x, h);
  check_weight(w_in, r.W, "w_in");
  const int N = w_in.size(0);
  TORCH_CHECK(N % 64 == 0, "gate and up in whole tiles");
  check_weight(w_down, N / 2, "w_down");
  TORCH_CHECK(w_down.size(0) == r.W);
  r.norm(w_post, "w_post"); r.norm(w_next, "w_next");
  auto st = cur_stream();
  auto act = torch::empty({r.T, N / 2}, h.options());
  if (glu_on_rows(r.T, r.W)) {
    TORCH_CHECK(launch_linear_rows(act.data_ptr(), bf(h), bf(w_in), nullptr, r.T, N, r.W, r.W, ROWS_CLAMPED, 1, (float)limit,
                                   (float)alpha, once, st) == 0, NO_LDS);
  } else {
    const Tensor y = at::linear(h, w_in);
    seq_launch_gated_act(act.data_ptr(), y.data_ptr(), bf(y, N / 2), r.T, N / 2, N, (float)limit, (float)alpha, 1.0f, 0, st);
  }
  const Tensor p = part(act, w_down, r.T, once, st);
  auto out = torch::empty_like(h);
  seq_launch_sandwich_rows(x.data_ptr<float>(), p.data_ptr<float>(), p.size(0), nullptr, 0, nullptr, nullptr,
                           w_post.data_ptr<float>(), w_next.data_ptr<float>(), out.data_ptr(), r.T, r.W, (float)eps, nullptr, 0, 0.0f, st);
  return out;
}
