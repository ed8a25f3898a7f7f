// PyTorch bindings for the kllms_amd gfx950 kernels (kllms_amd._C).
// Thin launch shims: shape/dtype checks, grid math, current-HIP-stream launch.

#include <torch/extension.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/HIPContext.h>
#include <c10/core/DeviceGuard.h>

#include "common.h"

// kernels (defined in the sibling .hip TUs)
extern "C" __global__ void rmsnorm_kernel(bf16_t*, const bf16_t*, const bf16_t*, int, float);
extern "C" __global__ void fused_add_rmsnorm_kernel(bf16_t*, const bf16_t*, bf16_t*, const bf16_t*, int, float);
extern "C" __global__ void silu_mul_kernel(bf16_t*, const bf16_t*, const bf16_t*, int64_t, int, int);
extern "C" __global__ void rope_kernel(bf16_t*, bf16_t*, const int64_t*, const float*, int, int, int, int, int);
extern "C" __global__ void store_kv_kernel(const bf16_t*, const bf16_t*, bf16_t*, bf16_t*, const int64_t*, int, int, int, int, int);
extern "C" __global__ void store_kv_fp8_kernel(const bf16_t*, const bf16_t*, unsigned char*, unsigned char*, float*, float*, const int64_t*, int, int, int, int, int);
extern "C" int attn_decode_splits(int B, int num_kv_heads, int gqa, int max_ctx, int fp8, int local, int joined);
extern "C" void launch_attn_decode(bf16_t*, float*, int*, int, const bf16_t*, const void*, const void*, const float*, const float*, const int*, const int*, const bf16_t*, int, float, int, int, int, int, int, int, int, int, int, hipStream_t);
extern "C" int launch_attn_prefill(bf16_t*, const bf16_t*, const bf16_t*, const bf16_t*, const int*, const int*, const int*, int, int, float, int, int, int, int, hipStream_t);
extern "C" int launch_attn_prefill_paged(bf16_t*, const bf16_t*, const bf16_t*, const bf16_t*, const int*, const int*, const int*, const int*, const int*, const int*, int, float, int, int, int, int, int, int, hipStream_t);
extern "C" void launch_attn_prefill_plan(int*, const int*, int, int, hipStream_t);
extern "C" int64_t sample_room(int B, int V, int masked);
extern "C" void launch_sample(int64_t*, float*, void*, const float*, const float*, const float*, const int*, const int64_t*, const int64_t*, const uint32_t*, int, int, float*, hipStream_t);
extern "C" __global__ void mfma_selftest_kernel(float*, const bf16_t*, const bf16_t*);

#define CHECK_BF16_CONTIG(t) \
  TORCH_CHECK((t).is_cuda() && (t).is_contiguous() && (t).scalar_type() == at::kBFloat16, #t " must be contiguous bf16 on GPU")

// [T, H, D] activation views: head/dim dims packed, token stride free (so the
// fused-QKV splits need no .contiguous() copies)
#define CHECK_KV_CACHE(t) \
  TORCH_CHECK((t).is_cuda() && (t).is_contiguous() && \
              ((t).scalar_type() == at::kBFloat16 || (t).scalar_type() == at::kFloat8_e4m3fn), \
              #t " must be a contiguous bf16 or fp8-e4m3 KV cache on GPU")

#define CHECK_BF16_ROWS(t) \
  TORCH_CHECK((t).is_cuda() && (t).scalar_type() == at::kBFloat16 && (t).dim() == 3 && \
              (t).stride(2) == 1 && (t).stride(1) == (t).size(2), #t " must be a bf16 [T,H,D] row view")

static inline hipStream_t cur_stream() {
  return at::hip::getCurrentHIPStream().stream();
}

static bf16_t* bf(torch::Tensor& t) { return reinterpret_cast<bf16_t*>(t.data_ptr()); }
static const bf16_t* cbf(const torch::Tensor& t) { return reinterpret_cast<const bf16_t*>(t.data_ptr()); }

void rmsnorm(torch::Tensor out, torch::Tensor in, torch::Tensor weight, double eps) {
  CHECK_BF16_CONTIG(out); CHECK_BF16_CONTIG(in); CHECK_BF16_CONTIG(weight);
  const int n = in.size(-1);
  TORCH_CHECK(n % 8 == 0, "hidden size must be a multiple of 8");
  const int rows = in.numel() / n;
  hipLaunchKernelGGL(rmsnorm_kernel, dim3(rows), dim3(256), 0, cur_stream(),
                     bf(out), cbf(in), cbf(weight), n, (float)eps);
}

void fused_add_rmsnorm(torch::Tensor out, torch::Tensor x, torch::Tensor residual,
                       torch::Tensor weight, double eps) {
  CHECK_BF16_CONTIG(out); CHECK_BF16_CONTIG(x); CHECK_BF16_CONTIG(residual); CHECK_BF16_CONTIG(weight);
  const int n = x.size(-1);
  TORCH_CHECK(n % 8 == 0, "hidden size must be a multiple of 8");
  const int rows = x.numel() / n;
  hipLaunchKernelGGL(fused_add_rmsnorm_kernel, dim3(rows), dim3(256), 0, cur_stream(),
                     bf(out), cbf(x), bf(residual), cbf(weight), n, (float)eps);
}

void silu_mul(torch::Tensor out, torch::Tensor gate, torch::Tensor up) {
  CHECK_BF16_CONTIG(out);
  TORCH_CHECK(gate.is_cuda() && gate.scalar_type() == at::kBFloat16 && gate.dim() == 2 &&
              gate.stride(1) == 1, "gate must be a bf16 [T, I] row view");
  TORCH_CHECK(up.sizes() == gate.sizes() && up.stride(0) == gate.stride(0) && up.stride(1) == 1);
  const int64_t ncols = gate.size(1);
  TORCH_CHECK(ncols % 8 == 0 && gate.stride(0) % 8 == 0);
  const int64_t nvec = gate.numel() / 8;
  const int grid = (int)std::min<int64_t>((nvec + 255) / 256, 2048);
  hipLaunchKernelGGL(silu_mul_kernel, dim3(grid), dim3(256), 0, cur_stream(),
                     bf(out), cbf(gate), cbf(up), nvec, (int)(ncols / 8), (int)(gate.stride(0) / 8));
}

void rope_inplace(torch::Tensor q, torch::Tensor k, torch::Tensor positions, torch::Tensor cos_sin) {
  CHECK_BF16_ROWS(q); CHECK_BF16_ROWS(k);
  TORCH_CHECK(positions.scalar_type() == at::kLong && cos_sin.scalar_type() == at::kFloat);
  const int T = q.size(0), H = q.size(1), D = q.size(2), KVH = k.size(1);
  hipLaunchKernelGGL(rope_kernel, dim3(T, H + KVH), dim3(D / 2), 0, cur_stream(),
                     bf(q), bf(k), positions.data_ptr<int64_t>(), cos_sin.data_ptr<float>(),
                     H, KVH, D, (int)q.stride(0), (int)k.stride(0));
}

void store_kv(torch::Tensor k, torch::Tensor v, torch::Tensor k_cache, torch::Tensor v_cache,
              torch::Tensor slot_mapping, torch::Tensor k_scale, torch::Tensor v_scale) {
  CHECK_BF16_ROWS(k); CHECK_BF16_ROWS(v); CHECK_KV_CACHE(k_cache); CHECK_KV_CACHE(v_cache);
  TORCH_CHECK(k.stride(0) == v.stride(0), "k/v must share the token stride");
  const int T = k.size(0), KVH = k.size(1), D = k.size(2);
  const int BS = k_cache.size(2);
  if (k_cache.scalar_type() == at::kFloat8_e4m3fn) {
    // per-row quantization: one wave per (token, head) row, 4 waves/block
    TORCH_CHECK(k_scale.numel() == k_cache.size(0) * KVH * BS && k_scale.is_contiguous() &&
                    k_scale.scalar_type() == at::kFloat && v_scale.numel() == k_scale.numel(),
                "fp8 store_kv requires [NB, KVH, BS] fp32 k_scale/v_scale");
    const int64_t rows = (int64_t)T * KVH;
    const int grid = (int)std::min<int64_t>((rows + 3) / 4, 2048);
    hipLaunchKernelGGL(store_kv_fp8_kernel, dim3(grid), dim3(256), 0, cur_stream(),
                       cbf(k), cbf(v),
                       reinterpret_cast<unsigned char*>(k_cache.data_ptr()),
                       reinterpret_cast<unsigned char*>(v_cache.data_ptr()),
                       k_scale.data_ptr<float>(), v_scale.data_ptr<float>(),
                       slot_mapping.data_ptr<int64_t>(), T, KVH, D, BS, (int)k.stride(0));
  } else {
    const int64_t total = (int64_t)T * KVH * (D / 8);
    const int grid = (int)std::min<int64_t>((total + 255) / 256, 2048);
    hipLaunchKernelGGL(store_kv_kernel, dim3(grid), dim3(256), 0, cur_stream(),
                       cbf(k), cbf(v), bf(k_cache), bf(v_cache),
                       slot_mapping.data_ptr<int64_t>(), T, KVH, D, BS, (int)k.stride(0));
  }
}

extern "C" void launch_rope_store(bf16_t* q, bf16_t* k, const bf16_t* v, const int64_t* positions,
                                  const float* cos_sin, void* k_cache, void* v_cache, float* k_scale, float* v_scale,
                                  const int64_t* slots, int T, int H, int G, int q_stride, int kv_stride,
                                  int block_size, int fp8, hipStream_t stream);

// rope_inplace and store_kv of rows of head size 128 in one launch; views of 16-byte aligned rows
void rope_store(torch::Tensor q, torch::Tensor k, torch::Tensor v, torch::Tensor positions, torch::Tensor cos_sin,
                torch::Tensor k_cache, torch::Tensor v_cache, torch::Tensor slots, torch::Tensor k_scale,
                torch::Tensor v_scale) {
  CHECK_BF16_ROWS(q); CHECK_BF16_ROWS(k); CHECK_BF16_ROWS(v); CHECK_KV_CACHE(k_cache); CHECK_KV_CACHE(v_cache);
  const int T = q.size(0), H = q.size(1), G = k.size(1), BS = k_cache.size(2);
  TORCH_CHECK(q.size(2) == 128 && k.size(2) == 128 && v.sizes() == k.sizes() && k.size(0) == T &&
                  k.stride(0) == v.stride(0) && k_cache.size(1) == G && k_cache.size(3) == 128 &&
                  v_cache.sizes() == k_cache.sizes() && v_cache.scalar_type() == k_cache.scalar_type(),
              "rope_store: sizes");
  for (const auto& t : {q, k, v})
    TORCH_CHECK(t.stride(0) % 8 == 0 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0, "rope_store: alignment");
  TORCH_CHECK(positions.scalar_type() == at::kLong && positions.is_contiguous() && positions.numel() == T &&
                  slots.scalar_type() == at::kLong && slots.is_contiguous() && slots.numel() == T &&
                  cos_sin.scalar_type() == at::kFloat && cos_sin.is_contiguous() && cos_sin.size(-1) == 128,
              "rope_store: positions, slots or angles");
  const int fp8 = k_cache.scalar_type() == at::kFloat8_e4m3fn ? 1 : 0;
  if (fp8)
    TORCH_CHECK(k_scale.numel() == k_cache.size(0) * G * BS && k_scale.is_contiguous() &&
                    k_scale.scalar_type() == at::kFloat && v_scale.numel() == k_scale.numel() &&
                    v_scale.is_contiguous() && v_scale.scalar_type() == at::kFloat,
                "fp8 rope_store requires [NB, KVH, BS] fp32 k_scale/v_scale");
  if (T == 0) return;
  launch_rope_store(bf(q), bf(k), cbf(v), positions.data_ptr<int64_t>(), cos_sin.data_ptr<float>(), k_cache.data_ptr(),
                    v_cache.data_ptr(), fp8 ? k_scale.data_ptr<float>() : nullptr,
                    fp8 ? v_scale.data_ptr<float>() : nullptr, slots.data_ptr<int64_t>(), T, H, G, (int)q.stride(0),
                    (int)k.stride(0), BS, fp8, cur_stream());
}

// mask_size: -1 for plain decode rows, from 0 (plain causal) on for those of a block-local layer
void attn_decode_paged(torch::Tensor out, torch::Tensor q, torch::Tensor k_cache,
                       torch::Tensor v_cache, torch::Tensor block_tables,
                       torch::Tensor context_lens, double scale,
                       torch::Tensor k_scale, torch::Tensor v_scale, torch::Tensor gate, int64_t mask_size, std::optional<torch::Tensor> arrived) {
  CHECK_BF16_CONTIG(out); CHECK_BF16_ROWS(q); CHECK_KV_CACHE(k_cache); CHECK_KV_CACHE(v_cache);
  const int B = q.size(0), H = q.size(1), D = q.size(2);
  const int KVH = k_cache.size(1), BS = k_cache.size(2);
  TORCH_CHECK(D == 128, "attn_decode: head_dim must be 128");
  TORCH_CHECK(H % KVH == 0, "attn_decode: H must be a multiple of KVH");
  TORCH_CHECK(H / KVH == 1 || H / KVH == 2 || H / KVH == 4 || H / KVH == 8,
              "attn_decode: GQA group must be 1, 2, 4 or 8");
  const int gqa = H / KVH;
  const int max_blocks = block_tables.size(1);
  TORCH_CHECK((int64_t)k_cache.size(0) * KVH * BS < (1LL << 31), "attn_decode: cache rows exceed 32-bit indexing");
  if (B == 0) return;
  if (max_blocks == 0) {       // every context is empty: the kernel looks at a row's first block before its length
    out.zero_();
    return;
  }
  // 16-byte query loads
  if (q.stride(0) % 8 != 0 || reinterpret_cast<uintptr_t>(q.data_ptr()) % 16 != 0) q = q.contiguous();
  if (gate.numel() > 0)
    TORCH_CHECK(gate.is_cuda() && gate.scalar_type() == at::kBFloat16 && gate.dim() == 2 && gate.size(0) == B &&
                    gate.size(1) == H && gate.stride(1) == 1, "gate must be a bf16 [B, H] row view");
  const int64_t longest = mask_size > 0 ? std::min<int64_t>(mask_size, (int64_t)max_blocks * BS) : (int64_t)max_blocks * BS;
  const int longest32 = (int)std::min<int64_t>(longest, INT32_MAX);
  const int splits = attn_decode_splits(B, KVH, gqa, longest32, k_cache.scalar_type() == at::kFloat8_e4m3fn, mask_size >= 0,
                                        arrived.has_value());
  int apart = 1;
  if (arrived) {
    TORCH_CHECK(arrived->is_cuda() && arrived->is_contiguous() && arrived->scalar_type() == at::kInt &&
                    arrived->numel() >= (int64_t)B * KVH, "arrived: an int32 zero for each row and kv head");
    apart = (int)std::min<int64_t>(arrived->numel() / ((int64_t)B * KVH), 32);
  }
  auto partials = torch::empty({splits > 1 ? (int64_t)B * KVH * splits * gqa * 130 : 0},
                               torch::dtype(torch::kFloat).device(q.device()));
  const int cache_fp8 = k_cache.scalar_type() == at::kFloat8_e4m3fn ? 1 : 0;
  if (cache_fp8) {
    TORCH_CHECK(k_scale.numel() == k_cache.size(0) * KVH * BS && k_scale.is_contiguous() &&
                    k_scale.scalar_type() == at::kFloat && v_scale.numel() == k_scale.numel(),
                "fp8 attn_decode requires [NB, KVH, BS] fp32 k_scale/v_scale");
  }
  launch_attn_decode(
      bf(out), partials.data_ptr<float>(), arrived ? arrived->data_ptr<int>() : nullptr, apart, cbf(q), k_cache.data_ptr(), v_cache.data_ptr(),
      cache_fp8 ? k_scale.data_ptr<float>() : nullptr,
      cache_fp8 ? v_scale.data_ptr<float>() : nullptr,
      block_tables.data_ptr<int>(), context_lens.data_ptr<int>(), gate.numel() ? cbf(gate) : nullptr,
      gate.numel() ? (int)gate.stride(0) : 0, (float)scale, H, KVH, BS, max_blocks, longest32, (int)q.stride(0), B,
      cache_fp8, (int)mask_size, cur_stream());
}

static bool rows_aligned(const torch::Tensor& t) {  // 16-byte row loads
  return t.stride(0) % 8 == 0 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

// rows of their own: also of a contiguous tensor that begins off 16 bytes, which contiguous() gives as it is
static torch::Tensor own_rows(const torch::Tensor& t) { return t.clone(at::MemoryFormat::Contiguous); }

// groups of 256 rows of the packed sequences cu [n + 1] over T rows: [3, G] (start, length, first row)
torch::Tensor attn_prefill_plan(torch::Tensor cu, int64_t T) {
  TORCH_CHECK(cu.is_cuda() && cu.is_contiguous() && cu.scalar_type() == at::kInt && cu.numel() >= 1);
  const int n = cu.numel() - 1;
  const int G = (int)(T / 256) + n;
  auto plan = torch::empty({3, G}, cu.options());
  if (G > 0) launch_attn_prefill_plan(plan.data_ptr<int>(), cu.data_ptr<int>(), n, G, cur_stream());
  return plan;
}

void attn_prefill(torch::Tensor out, torch::Tensor q, torch::Tensor k, torch::Tensor v,
                  torch::Tensor plan, double scale) {
  CHECK_BF16_CONTIG(out); CHECK_BF16_ROWS(q); CHECK_BF16_ROWS(k); CHECK_BF16_ROWS(v);
  const int H = q.size(1), D = q.size(2), KVH = k.size(1);
  TORCH_CHECK(D == 128, "attn_prefill: head_dim must be 128");
  TORCH_CHECK(H % KVH == 0, "attn_prefill: H must be a multiple of KVH");
  TORCH_CHECK(k.stride(0) == v.stride(0), "k/v must share the token stride");
  TORCH_CHECK(plan.is_cuda() && plan.is_contiguous() && plan.scalar_type() == at::kInt && plan.dim() == 2 &&
                  plan.size(0) == 3, "plan must come from attn_prefill_plan");
  const int G = plan.size(1);
  if (G == 0) return;
  if (!rows_aligned(q)) q = own_rows(q);
  if (!rows_aligned(k) || !rows_aligned(v)) { k = own_rows(k); v = own_rows(v); }
  const int* p = plan.data_ptr<int>();
  TORCH_CHECK(launch_attn_prefill(bf(out), cbf(q), cbf(k), cbf(v), p, p + G, p + 2 * G, 1, G, (float)scale, H, KVH,
                                  (int)q.stride(0), (int)k.stride(0), cur_stream()) == 0,
              "attn_prefill: 128 KB of LDS are not available");
}

// rows of segments against the paged cache (bf16): plan [4, G] int32 (first row, rows, first row within the
// segment, segment), tables [n, MAXB], pos [n] = position of each segment's first row. The segments' own keys and
// values are in the cache already. rows: of the plan's groups, 64 or 256.
void attn_prefill_paged(torch::Tensor out, torch::Tensor q, torch::Tensor k_cache, torch::Tensor v_cache,
                        torch::Tensor plan, torch::Tensor tables, torch::Tensor pos, double scale, int64_t rows) {
  CHECK_BF16_CONTIG(out); CHECK_BF16_ROWS(q); CHECK_BF16_CONTIG(k_cache); CHECK_BF16_CONTIG(v_cache);
  const int H = q.size(1), KVH = k_cache.size(1), BS = k_cache.size(2);
  TORCH_CHECK(q.size(2) == 128 && k_cache.size(3) == 128 && v_cache.sizes() == k_cache.sizes() && H % KVH == 0,
              "attn_prefill_paged: head size 128, whole groups");
  TORCH_CHECK(plan.is_cuda() && plan.is_contiguous() && plan.scalar_type() == at::kInt && plan.dim() == 2 &&
                  plan.size(0) == 4 && tables.is_cuda() && tables.is_contiguous() && tables.scalar_type() == at::kInt &&
                  tables.dim() == 2 && pos.is_cuda() && pos.is_contiguous() && pos.scalar_type() == at::kInt &&
                  pos.numel() == tables.size(0), "attn_prefill_paged: plan, tables or positions");
  TORCH_CHECK(rows == 64 || rows == 256, "attn_prefill_paged: groups of 64 or 256 rows");
  const int G = plan.size(1);
  if (G == 0) return;
  if (!rows_aligned(q)) q = own_rows(q);
  if (!rows_aligned(k_cache)) k_cache = own_rows(k_cache);
  if (!rows_aligned(v_cache)) v_cache = own_rows(v_cache);
  const int* p = plan.data_ptr<int>();
  TORCH_CHECK(launch_attn_prefill_paged(bf(out), cbf(q), cbf(k_cache), cbf(v_cache), p, p + G, p + 2 * G, p + 3 * G,
                                        tables.data_ptr<int>(), pos.data_ptr<int>(), G, (float)scale, H, KVH, (int)q.stride(0),
                                        BS, (int)tables.size(1), (int)rows, cur_stream()) == 0,
              "attn_prefill_paged: 128 KB of LDS are not available");
}

// (tokens, logprobs). The results are allocated here: 16 rows take 8.8 us on the device, and from Python the two allocations
// kept it waiting
std::tuple<torch::Tensor, torch::Tensor> sample(torch::Tensor logits, torch::Tensor temperatures, torch::Tensor top_ps,
                                                torch::Tensor top_ks, torch::Tensor seeds, torch::Tensor steps,
                                                std::optional<torch::Tensor> mask, std::optional<torch::Tensor> dbg) {
  TORCH_CHECK(logits.is_cuda() && logits.is_contiguous() && logits.scalar_type() == at::kFloat);
  const int B = logits.size(0), V = logits.size(1);
  const auto whole = torch::dtype(torch::kLong).device(logits.device());
  auto tokens = torch::empty({B}, whole), logprobs = torch::empty({B}, logits.options());
  const uint32_t* mptr = mask && mask->numel() > 0 ? reinterpret_cast<const uint32_t*>(mask->data_ptr<int>()) : nullptr;
  if (B == 0 || V == 0) return {tokens, logprobs};
  // per-slice results and lists
  auto parts = torch::empty({sample_room(B, V, mptr != nullptr)}, whole);
  launch_sample(tokens.data_ptr<int64_t>(), logprobs.data_ptr<float>(), parts.data_ptr(),
                logits.data_ptr<float>(), temperatures.data_ptr<float>(), top_ps.data_ptr<float>(),
                top_ks.data_ptr<int>(), seeds.data_ptr<int64_t>(), steps.data_ptr<int64_t>(), mptr,
                B, V, dbg && dbg->numel() ? dbg->data_ptr<float>() : nullptr, cur_stream());
  return {tokens, logprobs};
}

torch::Tensor mfma_selftest(torch::Tensor A, torch::Tensor B) {
  // D[32,32] = A[32,16] x B[16,32], verifying the fragment maps the attention
  // kernel assumes for v_mfma_f32_32x32x16_bf16.
  CHECK_BF16_CONTIG(A); CHECK_BF16_CONTIG(B);
  auto D = torch::empty({32, 32}, torch::dtype(torch::kFloat).device(A.device()));
  hipLaunchKernelGGL(mfma_selftest_kernel, dim3(1), dim3(64), 0, cur_stream(),
                     D.data_ptr<float>(), cbf(A), cbf(B));
  return D;
}

extern "C" void launch_one_shot_allreduce(const void* const* srcs, void* const* dsts,
                                          int n_peers, long numel, int write_all,
                                          hipStream_t stream);

void one_shot_allreduce(std::vector<torch::Tensor> bufs) {
  // In-place sum across up to 8 same-shaped bf16 buffers (single-GPU
  // simulation of the one-shot xGMI all-reduce: every "peer" buffer ends
  // holding the fp32-accumulated sum). Multi-GPU wiring (IPC-mapped peer
  // pointers, write_all=0) is round-2 work — docs/ROADMAP.md item 1.
  TORCH_CHECK(!bufs.empty() && bufs.size() <= 8, "1..8 peer buffers");
  const auto numel = bufs[0].numel();
  TORCH_CHECK(numel % 8 == 0, "numel must be a multiple of 8 (16B vector path)");
  const void* srcs[8];
  void* dsts[8];
  for (size_t r = 0; r < bufs.size(); ++r) {
    CHECK_BF16_CONTIG(bufs[r]);
    TORCH_CHECK(bufs[r].numel() == numel, "peer buffers must match in size");
    srcs[r] = bufs[r].data_ptr();
    dsts[r] = bufs[r].data_ptr();
  }
  launch_one_shot_allreduce(srcs, dsts, (int)bufs.size(), (long)numel, /*write_all=*/1,
                            cur_stream());
}

// --- grouped MoE expert GEMMs (moe.hip) --------------------------------------
extern "C" int launch_moe_gateup(void* act, const void* x, const void* w, const int* sorted_ids, const int* offsets,
                                 const void* zeros, int S, int E, int IN, int K, hipStream_t stream);
extern "C" int launch_moe_down(void* y, const void* act, const void* w, const int* offsets, float* part, int* count,
                               int S, int E, int H, int IN, hipStream_t stream);
extern "C" int64_t moe_down_room(int S, int E, int H, int IN, int* zeros);
extern "C" void launch_moe_sort(int* ids, int* pos, int* offsets, const int64_t* topi, int P, int k, int E,
                                hipStream_t stream);
extern "C" int moe_route_groups(int T);
extern "C" void launch_moe_route(int* topi, float* topw, int* rank, int* counts, const void* x, const void* gate, int T, int H,
                                 int64_t x_stride, int E, int k, hipStream_t stream);
extern "C" void launch_moe_place(int* ids, int* pos, int* offsets, int* zeros, int n_zeros, const int* topi, const int* rank,
                                 const int* counts, int T, int k, int E, hipStream_t stream);
extern "C" void launch_moe_combine(void* out, const void* y, const float* weights, const int* pos, int T, int k,
                                   int H, hipStream_t stream);

// what the products copy to LDS and store in 16-byte pieces: a view that does not begin on such a piece is copied
static torch::Tensor on_16_bytes(const torch::Tensor& t) {
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 ? t.clone() : t;
}

void moe_gateup(torch::Tensor act, torch::Tensor x, torch::Tensor w,
                torch::Tensor sorted_ids, torch::Tensor offsets, torch::Tensor zeros) {
  CHECK_BF16_CONTIG(act); CHECK_BF16_CONTIG(x); CHECK_BF16_CONTIG(w); CHECK_BF16_CONTIG(zeros);
  TORCH_CHECK(sorted_ids.scalar_type() == at::kInt && offsets.scalar_type() == at::kInt &&
                  sorted_ids.is_contiguous() && offsets.is_contiguous(), "routing tensors must be int32");
  const int E = w.size(0);
  const int IN = w.size(1) / 2;
  const int K = w.size(2);
  TORCH_CHECK(IN % 64 == 0 && K % 64 == 0, "IN % 64, K % 64 required");
  TORCH_CHECK(act.size(1) == IN && x.size(1) == K && zeros.numel() >= K);
  TORCH_CHECK(sorted_ids.numel() >= act.size(0), "one id per sorted row");
  TORCH_CHECK(offsets.numel() == E + 1);
  TORCH_CHECK(K < (1 << 24), "moe_gateup: a row of a tile's weights has a 32-bit offset");
  if (act.size(0) == 0) return;
  x = on_16_bytes(x), w = on_16_bytes(w), zeros = on_16_bytes(zeros);
  auto out = on_16_bytes(act);
  TORCH_CHECK(launch_moe_gateup(out.data_ptr(), x.data_ptr(), w.data_ptr(), sorted_ids.data_ptr<int>(),
                                offsets.data_ptr<int>(), zeros.data_ptr(), (int)act.size(0), E, IN, K,
                                cur_stream()) == 0, "moe_gateup: 160 KB of LDS are not available");
  if (!out.is_same(act)) act.copy_(out);
}

#define MOE_DOWN_COUNTERS 256

// cleared: MOE_DOWN_COUNTERS int32 zeros that this call uses up, or nothing: it makes its own
void moe_down(torch::Tensor y, torch::Tensor act, torch::Tensor w, torch::Tensor offsets, std::optional<torch::Tensor> cleared) {
  CHECK_BF16_CONTIG(y); CHECK_BF16_CONTIG(act); CHECK_BF16_CONTIG(w);
  const int E = w.size(0);
  const int H = w.size(1);
  const int IN = w.size(2);
  TORCH_CHECK(H % 64 == 0 && IN % 64 == 0, "H % 64, IN % 64 required");
  TORCH_CHECK(y.size(1) == H && act.size(1) == IN && y.size(0) >= act.size(0));
  TORCH_CHECK(offsets.numel() == E + 1 && offsets.scalar_type() == at::kInt && offsets.is_contiguous());
  TORCH_CHECK(IN < (1 << 24), "moe_down: a row of a tile's weights has a 32-bit offset");
  if (act.size(0) == 0) return;
  act = on_16_bytes(act), w = on_16_bytes(w);
  auto out = on_16_bytes(y);
  // partial sums and counters of tiles that are worked on in shares
  int zeros = 0;
  const int64_t room = moe_down_room(act.size(0), E, H, IN, &zeros);
  torch::Tensor part, count;
  if (room) {
    part = torch::empty({room}, act.options().dtype(torch::kFloat));
    if (cleared) {
      TORCH_CHECK(cleared->is_cuda() && cleared->scalar_type() == at::kInt && cleared->is_contiguous() &&
                      cleared->numel() >= zeros, "moe_down: counters");
      count = *cleared;
    } else {
      count = torch::zeros({zeros}, act.options().dtype(torch::kInt));
    }
  }
  TORCH_CHECK(launch_moe_down(out.data_ptr(), act.data_ptr(), w.data_ptr(), offsets.data_ptr<int>(),
                              room ? part.data_ptr<float>() : nullptr, room ? count.data_ptr<int>() : nullptr, (int)act.size(0), E, H, IN,
                              cur_stream()) == 0, "moe_down: 160 KB of LDS are not available");
  if (!out.is_same(y)) y.copy_(out);
}

// --- products of many rows (linear_tiles.hip) ---------------------------------
extern "C" int linear_tiles_rows(int64_t M, int64_t N, int64_t K, int act);
extern "C" int64_t linear_tiles_room(int mj, int* zeros);
extern "C" int launch_linear_tiles(void* out, const void* x, const void* w, const void* bias, float* part, int* count, int M,
                                   int N, int K, int act, int mj, float limit, float alpha, hipStream_t stream);

// act 0: x [M, K] @ w [N, K]^T + bias (or an empty one); 1, 2: w [2 N, K], silu(gate) * up or the clamped form.
// mj: 32-row steps of a tile, 2 to 8; share: the last round's tiles are shared out over K
torch::Tensor linear_tiles(torch::Tensor x, torch::Tensor w, torch::Tensor bias, int act, int mj, bool share,
                           double limit, double alpha) {
  CHECK_BF16_CONTIG(x); CHECK_BF16_CONTIG(w);
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1) && x.device() == w.device(), "x [M, K], w [N, K]");
  TORCH_CHECK(act >= 0 && act <= 2 && mj >= 2 && mj <= 8, "linear_tiles: act 0 to 2, mj 2 to 8");
  const int64_t M = x.size(0), K = x.size(1), N = act ? w.size(0) / 2 : w.size(0);
  TORCH_CHECK(!act || w.size(0) % 2 == 0, "gate and up have the same rows");
  TORCH_CHECK(K % 64 == 0 && K > 0 && K < (1 << 24) && N % 8 == 0 && N > 0 && N < (1 << 30) && M < (1 << 30),
              "linear_tiles: K % 64, N % 8 required");
  TORCH_CHECK(((M + 63) / 64) * ((N + 127) / 128) < (1 << 27), "linear_tiles: too many tiles");
  const bool biased = bias.numel() > 0;
  if (biased) {
    CHECK_BF16_CONTIG(bias);
    TORCH_CHECK(act == 0 && bias.numel() == N && bias.device() == x.device(), "bias [N] of a plain product");
  }
  auto on_16 = [](const torch::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; };
  TORCH_CHECK(on_16(x) && on_16(w) && (!biased || on_16(bias)), "linear_tiles: operands begin on 16 bytes");
  // as the library: on the device of x, whatever the current one is
  const c10::DeviceGuard device(x.device());
  auto out = torch::empty({M, N}, x.options());
  if (M == 0) return out;
  torch::Tensor part, count;
  if (share) {
    int zeros = 0;
    part = torch::empty({linear_tiles_room(mj, &zeros)}, x.options().dtype(torch::kFloat));
    count = torch::zeros({zeros}, x.options().dtype(torch::kInt));
  }
  TORCH_CHECK(launch_linear_tiles(out.data_ptr(), x.data_ptr(), w.data_ptr(), biased ? bias.data_ptr() : nullptr,
                                  share ? part.data_ptr<float>() : nullptr, share ? count.data_ptr<int>() : nullptr, M, N, K,
                                  act, mj, limit, alpha, cur_stream()) == 0,
              "linear_tiles: 160 KB of LDS are not available");
  return out;
}

// Whether nothing but the values of a tensor is wanted: no subclass, transform or gradient looks on
static bool plain_values(const torch::Tensor& t) {
  static const c10::DispatchKeySet others({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot,
                                           c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                           c10::DispatchKey::FuncTorchVmapMode, c10::DispatchKey::Batched,
                                           c10::DispatchKey::VmapMode, c10::DispatchKey::Functionalize,
                                           c10::DispatchKey::FuncTorchDynamicLayerFrontMode,
                                           c10::DispatchKey::FuncTorchDynamicLayerBackMode});
  const auto keys = t.key_set() | c10::impl::tls_local_dispatch_key_set().included_;
  return !keys.has_any(others) && !(at::GradMode::is_enabled() && t.requires_grad()) && !t._fw_grad(0).defined();
}

// mj of linear_tiles, + 16 for shares, where it takes the call and is the faster side of linear_tiles_rows; 0: the library's
int64_t linear_tiles_pick(const torch::Tensor& x, const torch::Tensor& w, const std::optional<torch::Tensor>& bias,
                          int64_t act) {
  if (x.dim() != 2 || w.dim() != 2 || x.size(0) <= 128 || !x.is_cuda() || x.device() != w.device() ||
      x.scalar_type() != at::kBFloat16 || w.scalar_type() != at::kBFloat16)
    return 0;
  if (!plain_values(x) || !plain_values(w) || torch::jit::tracer::isTracing()) return 0;
  if (at::autocast::is_autocast_enabled(at::kCUDA)) return 0;      // the library's product has autocast's type
  const int64_t M = x.size(0), K = x.size(1), N = act ? w.size(0) / 2 : w.size(0);
  auto on_16 = [](const torch::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; };
  if (K % 64 || K == 0 || K >= 1 << 24 || N % 8 || N == 0 || w.size(1) != K || std::max(M, N) >= 1 << 30 ||
      !x.is_contiguous() || !w.is_contiguous() || !on_16(x) || !on_16(w) || M * N >= (int64_t)1 << 38 ||
      (act && w.size(0) % 2))
    return 0;
  if (bias && !(bias->scalar_type() == at::kBFloat16 && bias->device() == x.device() && bias->dim() == 1 &&
                bias->size(0) == N && bias->is_contiguous() && on_16(*bias) && plain_values(*bias)))
    return 0;
  return linear_tiles_rows(M, N, K, (int)act);
}

// linear_tiles where linear_tiles_pick takes the call, else nothing. One call: from Python the checks alone are 5 us
std::optional<torch::Tensor> linear_tiles_try(torch::Tensor x, torch::Tensor w, std::optional<torch::Tensor> bias, int64_t act,
                                              double limit, double alpha) {
  const int64_t mj = linear_tiles_pick(x, w, bias, act);
  if (!mj) return std::nullopt;
  return linear_tiles(x, w, bias ? *bias : x.new_empty({0}), (int)act, mj & 15, mj > 15, limit, alpha);
}

// topi [T, k] int64 -> (ids [T * k] token of each sorted place, pos [T, k] sorted place of each pair,
// offsets [E + 1]); a pair without an expert of 0..E-1 gets pos -1
std::vector<torch::Tensor> moe_sort(torch::Tensor topi, int64_t E) {
  TORCH_CHECK(topi.is_cuda() && topi.is_contiguous() && topi.scalar_type() == at::kLong && topi.dim() == 2);
  TORCH_CHECK(E >= 1 && E <= 4096 && topi.numel() < (1LL << 31), "moe_sort: sizes");
  const int P = topi.numel(), k = topi.size(1);
  auto i32 = topi.options().dtype(torch::kInt);
  auto ids = torch::empty({P}, i32), pos = torch::empty({topi.size(0), k}, i32), offsets = torch::empty({E + 1}, i32);
  launch_moe_sort(ids.data_ptr<int>(), pos.data_ptr<int>(), offsets.data_ptr<int>(), topi.data_ptr<int64_t>(), P,
                  k > 0 ? k : 1, (int)E, cur_stream());
  return {ids, pos, offsets};
}

// The k experts of each row of x by the router's weights gate [E, H] and their shares (moe_route_kernel), and where
// ``places`` asks for it what moe_sort gives for them: (topw [T, k] fp32, topi [T, k] int32), then (ids, pos, offsets,
// counters for moe_down). Nothing where the kernel does not take the call, or where more than its values is wanted.
std::optional<std::vector<torch::Tensor>> moe_route_try(torch::Tensor x, torch::Tensor gate, int64_t k, bool places) {
  if (x.dim() != 2 || gate.dim() != 2 || !x.is_cuda() || x.device() != gate.device() || x.scalar_type() != at::kBFloat16 ||
      gate.scalar_type() != at::kBFloat16 || !plain_values(x) || !plain_values(gate) || torch::jit::tracer::isTracing() ||
      at::autocast::is_autocast_enabled(at::kCUDA))
    return std::nullopt;
  const int64_t T = x.size(0), H = x.size(1), E = gate.size(0);
  if (T < 1 || T * k >= 1LL << 31 || H < 64 || H % 64 || H >= 1 << 24 || gate.size(1) != H || E < 1 || E > 32 || k < 1 || k > 8 || k > E ||
      x.stride(1) != 1 || !rows_aligned(x) || !gate.is_contiguous() || reinterpret_cast<uintptr_t>(gate.data_ptr()) % 16)
    return std::nullopt;
  const c10::DeviceGuard device(x.device());
  const int groups = moe_route_groups((int)T);
  auto i32 = x.options().dtype(torch::kInt);
  auto topw = torch::empty({T, k}, x.options().dtype(torch::kFloat)), topi = torch::empty({T, k}, i32);
  auto rank = torch::empty({T * k}, i32), counts = torch::empty({groups, E}, i32);
  launch_moe_route(topi.data_ptr<int>(), topw.data_ptr<float>(), rank.data_ptr<int>(), counts.data_ptr<int>(), x.data_ptr(),
                   gate.data_ptr(), (int)T, (int)H, x.stride(0), (int)E, (int)k, cur_stream());
  if (!places) return std::vector<torch::Tensor>{topw, topi};
  auto ids = torch::empty({T * k}, i32), pos = torch::empty({T, k}, i32), offsets = torch::empty({E + 1}, i32);
  auto cleared = torch::empty({MOE_DOWN_COUNTERS}, i32);
  launch_moe_place(ids.data_ptr<int>(), pos.data_ptr<int>(), offsets.data_ptr<int>(), cleared.data_ptr<int>(),
                   MOE_DOWN_COUNTERS, topi.data_ptr<int>(), rank.data_ptr<int>(), counts.data_ptr<int>(), (int)T, (int)k, (int)E,
                   cur_stream());
  return std::vector<torch::Tensor>{topw, topi, ids, pos, offsets, cleared};
}

torch::Tensor moe_combine(torch::Tensor y, torch::Tensor weights, torch::Tensor pos) {
  CHECK_BF16_CONTIG(y);
  TORCH_CHECK(weights.is_cuda() && weights.is_contiguous() && weights.scalar_type() == at::kFloat &&
                  pos.is_cuda() && pos.is_contiguous() && pos.scalar_type() == at::kInt && pos.dim() == 2 &&
                  weights.sizes() == pos.sizes() && y.dim() == 2 && y.size(1) % 8 == 0);
  auto out = torch::empty({pos.size(0), y.size(1)}, y.options());
  if (out.numel() == 0) return out;
  launch_moe_combine(out.data_ptr(), y.data_ptr(), weights.data_ptr<float>(), pos.data_ptr<int>(), (int)pos.size(0),
                     (int)pos.size(1), (int)y.size(1), cur_stream());
  return out;
}

// --- products of a few rows (linear_rows.hip) ---------------------------------
extern "C" int linear_rows_most(int form);
extern "C" int64_t linear_rows_strides();
extern "C" int launch_linear_rows(void* out, const bf16_t* x, const bf16_t* w, const bf16_t* bias, int M, int N,
                                   int K, int x_stride, int form, int splits, float limit, float alpha, bool once,
                                   hipStream_t stream);
extern "C" int linear_rows_splits(int M, int N, int K);

// form 0: fp32 sums [S, M, N]; 1: bf16 [M, N] (+ bias); 2: fp32 [M, N]; 3: silu(gate) * up of a fused
// [gate; up] matrix, bf16 [M, N / 2]. once: the weights of the caller's step do not stay in the caches until its next
torch::Tensor linear_rows(torch::Tensor x, torch::Tensor w, torch::Tensor bias, int64_t form, int64_t splits, bool once) {
  TORCH_CHECK(x.is_cuda() && x.scalar_type() == at::kBFloat16 && x.dim() == 2 && x.stride(1) == 1 &&
                  x.stride(0) % 8 == 0 && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0,
              "x must be a bf16 [M, K] row view, 16-byte aligned");
  CHECK_BF16_CONTIG(w);
  const int M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(form >= 0 && form <= 3 && (form != 3 || N % 64 == 0));
  TORCH_CHECK(w.dim() == 2 && w.size(1) == K && M >= 1 && M <= linear_rows_most((int)form) && K % 128 == 0 && N % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0,
              "linear_rows: M in 1..", linear_rows_most((int)form), ", K a multiple of 128, N of 16");
  TORCH_CHECK(bias.numel() == 0 || (form == 1 && bias.numel() == N && bias.is_contiguous() &&
                                    bias.scalar_type() == at::kBFloat16), "bias: bf16 [N], bf16 form only");
  if (x.stride(0) >= linear_rows_strides()) x = x.contiguous();    // one row is contiguous whatever its stride
  const int x_stride = M == 1 ? K : (int)x.stride(0);
  int S = 1;
  if (form == 0) S = splits > 0 ? (int)std::min<int64_t>(splits, K / 64) : linear_rows_splits(M, N, K);
  auto out = form == 0 ? torch::empty({S, M, N}, x.options().dtype(torch::kFloat))
           : form == 2 ? torch::empty({M, N}, x.options().dtype(torch::kFloat))
                       : torch::empty({M, form == 3 ? N / 2 : N}, x.options());
  TORCH_CHECK(launch_linear_rows(out.data_ptr(), cbf(x), cbf(w), bias.numel() ? cbf(bias) : nullptr, M, N, K,
                                 x_stride, (int)form, S, 0.0f, 0.0f, once, cur_stream()) == 0,
              "linear_rows: 160 KB of LDS are not available");
  return out;
}

// What linear_rows and the row-wise steps ask of weights. One call for a model's: from Python a question is 1 us
bool rows_weights_ok(const std::vector<torch::Tensor>& ws, const torch::Tensor& like) {
  for (const auto& w : ws)
    if (w.layout() != at::kStrided || w.device() != like.device() || w.scalar_type() != at::kBFloat16 || !plain_values(w) ||
        !w.is_contiguous() || reinterpret_cast<uintptr_t>(w.data_ptr()) % 16)
      return false;
  return true;
}

// --- row-wise steps of a decode step (decode_rows.hip) -------------------------
extern "C" void launch_add_norm_rows(bf16_t* out, bf16_t* residual, const float* part, const int64_t* ids,
                                     const bf16_t* table, const bf16_t* w, int S, int M, int n, int64_t vocab,
                                     float eps, int* unknown, int* clear, int clears, hipStream_t stream);
extern "C" void launch_rope_store_rows(bf16_t* q_out, const float* part, const bf16_t* bias, const int64_t* positions,
                                       const float* cos_sin, void* k_cache, void* v_cache, float* k_scale,
                                       float* v_scale, const int64_t* slots, int S, int M, int H, int G,
                                       int block_size, int fp8, hipStream_t stream);
extern "C" void launch_decode_inputs(int64_t* ids, int64_t* positions, int64_t* slots, int* ctx, int* tables,
                                     const int64_t* ids_in, const int64_t* positions_in, const int64_t* slots_in,
                                     const int* ctx_in, const int* tables_in, int B, int bs, int nb, int mb,
                                     int scratch_block, int block_size, hipStream_t stream);

// residual += split sums [S, M, n]; returns rms(residual) * weight
torch::Tensor add_norm_rows(torch::Tensor part, torch::Tensor residual, torch::Tensor weight, double eps) {
  CHECK_BF16_CONTIG(residual); CHECK_BF16_CONTIG(weight);
  TORCH_CHECK(part.is_cuda() && part.is_contiguous() && part.scalar_type() == at::kFloat && part.dim() == 3);
  const int S = part.size(0), M = part.size(1), n = part.size(2);
  TORCH_CHECK(residual.dim() == 2 && residual.size(0) == M && residual.size(1) == n && weight.numel() == n &&
                  n % 4 == 0 && n <= 16384 && S >= 1 && M >= 1, "add_norm_rows: sizes");
  auto out = torch::empty_like(residual);
  launch_add_norm_rows(bf(out), bf(residual), part.data_ptr<float>(), nullptr, nullptr, cbf(weight), S, M, n, 0,
                       (float)eps, nullptr, nullptr, 0, cur_stream());
  return out;
}

// (rms(table[ids]) * weight, table[ids]); an id outside the table gives a row of NaN and sets unknown (empty, or one
// int32 of pinned host memory). clear: int32 values that are zeroed beside
std::vector<torch::Tensor> embed_norm_rows(torch::Tensor ids, torch::Tensor table, torch::Tensor weight, double eps,
                                           torch::Tensor unknown, std::optional<torch::Tensor> clear) {
  CHECK_BF16_CONTIG(table); CHECK_BF16_CONTIG(weight);
  TORCH_CHECK(ids.is_cuda() && ids.is_contiguous() && ids.scalar_type() == at::kLong && ids.dim() == 1);
  const int M = ids.size(0), n = table.size(1);
  TORCH_CHECK(weight.numel() == n && n % 4 == 0 && n <= 16384 && M >= 1, "embed_norm_rows: sizes");
  TORCH_CHECK(unknown.numel() == 0 || (unknown.numel() == 1 && unknown.scalar_type() == at::kInt && unknown.is_pinned()),
              "unknown: one int32 of pinned host memory");
  TORCH_CHECK(!clear || (clear->is_cuda() && clear->is_contiguous() && clear->scalar_type() == at::kInt &&
                         clear->numel() <= INT32_MAX), "clear: int32 values");
  auto residual = torch::empty({M, n}, table.options());
  auto out = torch::empty_like(residual);
  launch_add_norm_rows(bf(out), bf(residual), nullptr, ids.data_ptr<int64_t>(), cbf(table), cbf(weight), 0, M, n,
                       table.size(0), (float)eps, unknown.numel() ? unknown.data_ptr<int>() : nullptr,
                       clear ? clear->data_ptr<int>() : nullptr, clear ? (int)clear->numel() : 0, cur_stream());
  return {out, residual};
}

// rotates q and k of the fused projection's split sums, stores k and v; returns q [M, H, 128]
torch::Tensor rope_store_rows(torch::Tensor part, torch::Tensor bias, int64_t H, torch::Tensor positions,
                              torch::Tensor cos_sin, torch::Tensor k_cache, torch::Tensor v_cache,
                              torch::Tensor slots, torch::Tensor k_scale, torch::Tensor v_scale) {
  CHECK_KV_CACHE(k_cache); CHECK_KV_CACHE(v_cache);
  TORCH_CHECK(part.is_cuda() && part.is_contiguous() && part.scalar_type() == at::kFloat && part.dim() == 3);
  const int S = part.size(0), M = part.size(1), G = k_cache.size(1), BS = k_cache.size(2);
  TORCH_CHECK(k_cache.size(3) == 128 && v_cache.sizes() == k_cache.sizes() &&
                  v_cache.scalar_type() == k_cache.scalar_type() && part.size(2) == (H + 2 * G) * 128 && S >= 1 &&
                  M >= 1, "rope_store_rows: sizes");
  TORCH_CHECK(positions.scalar_type() == at::kLong && positions.is_contiguous() && positions.numel() == M &&
                  slots.scalar_type() == at::kLong && slots.is_contiguous() && slots.numel() == M &&
                  cos_sin.scalar_type() == at::kFloat && cos_sin.is_contiguous() && cos_sin.size(-1) == 128,
              "rope_store_rows: positions, slots or angles");
  TORCH_CHECK(bias.numel() == 0 || (bias.scalar_type() == at::kBFloat16 && bias.is_contiguous() &&
                                    bias.numel() == part.size(2)), "rope_store_rows: bias");
  const int fp8 = k_cache.scalar_type() == at::kFloat8_e4m3fn ? 1 : 0;
  if (fp8)
    TORCH_CHECK(k_scale.numel() == k_cache.size(0) * G * BS && k_scale.is_contiguous() &&
                    k_scale.scalar_type() == at::kFloat && v_scale.numel() == k_scale.numel() &&
                    v_scale.is_contiguous() && v_scale.scalar_type() == at::kFloat,
                "fp8 rope_store_rows requires [NB, KVH, BS] fp32 k_scale/v_scale");
  auto q = torch::empty({M, H, 128}, part.options().dtype(torch::kBFloat16));
  launch_rope_store_rows(bf(q), part.data_ptr<float>(), bias.numel() ? cbf(bias) : nullptr,
                         positions.data_ptr<int64_t>(), cos_sin.data_ptr<float>(), k_cache.data_ptr(),
                         v_cache.data_ptr(), fp8 ? k_scale.data_ptr<float>() : nullptr,
                         fp8 ? v_scale.data_ptr<float>() : nullptr, slots.data_ptr<int64_t>(), S, M, (int)H, G, BS,
                         fp8, cur_stream());
  return q;
}

// fills the fixed buffers of a captured step of bs rows from B <= bs rows
void decode_inputs(torch::Tensor ids, torch::Tensor positions, torch::Tensor slots, torch::Tensor ctx,
                   torch::Tensor tables, torch::Tensor ids_in, torch::Tensor positions_in, torch::Tensor slots_in,
                   torch::Tensor ctx_in, torch::Tensor tables_in, int64_t scratch_block, int64_t block_size) {
  const int64_t bs = ids.numel(), B = ids_in.numel();
  for (const auto& t : {ids, positions, slots, ids_in, positions_in, slots_in})
    TORCH_CHECK(t.is_cuda() && t.is_contiguous() && t.scalar_type() == at::kLong, "decode_inputs: int64 rows");
  for (const auto& t : {ctx, ctx_in, tables, tables_in})
    TORCH_CHECK(t.is_cuda() && t.is_contiguous() && t.scalar_type() == at::kInt, "decode_inputs: int32 rows");
  TORCH_CHECK(B <= bs && bs >= 1 && positions.numel() == bs && slots.numel() == bs && ctx.numel() == bs &&
                  positions_in.numel() == B && slots_in.numel() == B && ctx_in.numel() == B && tables.dim() == 2 &&
                  tables.size(0) == bs && tables_in.dim() == 2 && tables_in.size(0) == B &&
                  tables_in.size(1) <= tables.size(1), "decode_inputs: sizes");
  launch_decode_inputs(ids.data_ptr<int64_t>(), positions.data_ptr<int64_t>(), slots.data_ptr<int64_t>(),
                       ctx.data_ptr<int>(), tables.data_ptr<int>(), ids_in.data_ptr<int64_t>(),
                       positions_in.data_ptr<int64_t>(), slots_in.data_ptr<int64_t>(), ctx_in.data_ptr<int>(),
                       tables_in.data_ptr<int>(), (int)B, (int)bs, (int)tables_in.size(1), (int)tables.size(1),
                       (int)scratch_block, (int)block_size, cur_stream());
}

// --- batched Levenshtein (levenshtein.hip) -----------------------------------
extern "C" void launch_levenshtein(int* out, const unsigned char* chars, const int* lens,
                                   const int* pi, const int* pj, long n_pairs,
                                   hipStream_t stream);

torch::Tensor levenshtein_pairs(torch::Tensor chars, torch::Tensor lens,
                                torch::Tensor pair_i, torch::Tensor pair_j) {
  TORCH_CHECK(chars.is_cuda() && chars.scalar_type() == at::kByte && chars.size(1) == 64 &&
              chars.is_contiguous(), "chars must be contiguous uint8 [N, 64] on GPU");
  TORCH_CHECK(lens.scalar_type() == at::kInt && pair_i.scalar_type() == at::kInt &&
              pair_j.scalar_type() == at::kInt);
  const long P = pair_i.numel();
  auto out = torch::empty({P}, torch::dtype(torch::kInt).device(chars.device()));
  launch_levenshtein(out.data_ptr<int>(),
                     chars.data_ptr<unsigned char>(), lens.data_ptr<int>(),
                     pair_i.data_ptr<int>(), pair_j.data_ptr<int>(), P, cur_stream());
  return out;
}

// --- hipIpc one-shot all-reduce (allreduce.hip) ------------------------------
extern "C" void* ipc_ar_create(int rank, int world, size_t max_bytes, unsigned char* handles_out);
extern "C" int ipc_ar_connect(void* ctx, const unsigned char* all_handles);
extern "C" int ipc_ar_run(void* ctx, const void* inp, void* out, long numel, hipStream_t stream);
extern "C" void ipc_ar_destroy(void* ctx);

std::pair<int64_t, py::bytes> ipc_allreduce_create(int rank, int world, int64_t max_bytes) {
  unsigned char handles[128];
  void* ctx = ipc_ar_create(rank, world, (size_t)max_bytes, handles);
  TORCH_CHECK(ctx != nullptr, "ipc_ar_create failed (see stderr)");
  return {reinterpret_cast<int64_t>(ctx), py::bytes(reinterpret_cast<char*>(handles), 128)};
}

void ipc_allreduce_connect(int64_t ctx, py::bytes all_handles) {
  std::string h = all_handles;
  TORCH_CHECK(h.size() % 128 == 0, "handle blob must be world*128 bytes");
  int rc = ipc_ar_connect(reinterpret_cast<void*>(ctx),
                          reinterpret_cast<const unsigned char*>(h.data()));
  TORCH_CHECK(rc == 0, "ipc_ar_connect failed (see stderr)");
}

void ipc_allreduce_run(int64_t ctx, torch::Tensor inp, torch::Tensor out) {
  CHECK_BF16_CONTIG(inp);
  CHECK_BF16_CONTIG(out);
  TORCH_CHECK(inp.numel() == out.numel(), "in/out size mismatch");
  int rc = ipc_ar_run(reinterpret_cast<void*>(ctx), inp.data_ptr(), out.data_ptr(),
                      (long)inp.numel(), cur_stream());
  TORCH_CHECK(rc == 0, "ipc_ar_run failed rc=", rc);
}

void ipc_allreduce_destroy(int64_t ctx) {
  ipc_ar_destroy(reinterpret_cast<void*>(ctx));
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("levenshtein_pairs", &levenshtein_pairs);
  m.def("linear_rows", &linear_rows, py::arg("x"), py::arg("w"), py::arg("bias"), py::arg("form"), py::arg("splits"),
        py::arg("once") = false);
  m.def("rows_weights_ok", &rows_weights_ok);
  m.def("add_norm_rows", &add_norm_rows);
  m.def("embed_norm_rows", &embed_norm_rows, py::arg("ids"), py::arg("table"), py::arg("weight"), py::arg("eps"),
        py::arg("unknown"), py::arg("clear") = py::none());
  m.def("rope_store_rows", &rope_store_rows);
  m.def("decode_inputs", &decode_inputs);
  m.def("linear_tiles", &linear_tiles);
  m.def("linear_tiles_rows", &linear_tiles_rows);
  m.def("linear_tiles_pick", &linear_tiles_pick);
  m.def("linear_tiles_try", &linear_tiles_try);
  m.def("moe_gateup", &moe_gateup);
  m.def("moe_down", &moe_down, py::arg("y"), py::arg("act"), py::arg("w"), py::arg("offsets"),
        py::arg("cleared") = std::nullopt);
  m.def("moe_route_try", &moe_route_try);
  m.def("moe_sort", &moe_sort);
  m.def("moe_combine", &moe_combine);
  m.def("ipc_allreduce_create", &ipc_allreduce_create);
  m.def("ipc_allreduce_connect", &ipc_allreduce_connect);
  m.def("ipc_allreduce_run", &ipc_allreduce_run);
  m.def("ipc_allreduce_destroy", &ipc_allreduce_destroy);
  m.def("rmsnorm", &rmsnorm);
  m.def("fused_add_rmsnorm", &fused_add_rmsnorm);
  m.def("silu_mul", &silu_mul);
  m.def("rope_inplace", &rope_inplace);
  m.def("store_kv", &store_kv);
  m.def("rope_store", &rope_store);
  // workgroups of a context at most, by rows, kv heads, heads of each, positions of the table, fp8, block-local, counters
  m.def("attn_decode_splits", &attn_decode_splits);
  m.def("attn_decode_paged", &attn_decode_paged, py::arg("out"), py::arg("q"), py::arg("k_cache"),
        py::arg("v_cache"), py::arg("block_tables"), py::arg("context_lens"), py::arg("scale"), py::arg("k_scale"),
        py::arg("v_scale"), py::arg("gate"), py::arg("mask_size") = -1, py::arg("arrived") = py::none());
  m.def("attn_prefill", &attn_prefill);
  m.def("attn_prefill_plan", &attn_prefill_plan);
  m.def("attn_prefill_paged", &attn_prefill_paged, py::arg("out"), py::arg("q"), py::arg("k_cache"), py::arg("v_cache"),
        py::arg("plan"), py::arg("tables"), py::arg("pos"), py::arg("scale"), py::arg("rows") = 256);
  m.def("sample", &sample);
  m.def("mfma_selftest", &mfma_selftest);
  m.def("one_shot_allreduce", &one_shot_allreduce);
}
