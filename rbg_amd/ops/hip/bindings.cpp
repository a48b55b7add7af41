// PyTorch bindings for the rbg_amd CDNA4 HIP kernels.
// Thin shape/dtype checks here; all math lives in the .hip translation units.
#include <torch/extension.h>
#include <ATen/core/CachingHostAllocator.h>
#include <ATen/hip/HIPContext.h>

#include <hip/hip_runtime.h>

#include <cstring>
#include <vector>

#include "decode_heads.h"
#include "gemm_bindings.h"
#include "prefill_plan.h"
#include "tile_bindings.h"

extern "C" {
void launch_rmsnorm(void*, void*, const void*, float, int, int, hipStream_t);
void launch_fused_add_rmsnorm(void*, void*, const void*, float, int, int,
                              hipStream_t);
void launch_add_rmsnorm_rows(void*, const void*, void*, const void*, float,
                             int, int, int, hipStream_t);
void launch_rope_heads(void*, void*, void*, const void*, int, const void*,
                       const void*, float, void*, void*, const void*,
                       const void*, const void*, int, int, int, int, int, int,
                       hipStream_t);
void launch_embed_rows(void*, const void*, const void*, long, int, int, bool,
                       hipStream_t);
void launch_silu_parts(void*, const void*, int, int, int, hipStream_t);
void launch_silu_mul(void*, const void*, int, int, hipStream_t);
void launch_rope_store_kv(void*, void*, const void*, void*, void*,
                          const void*, const void*, const void*, int, int,
                          int, int, int, int, int, hipStream_t);
void launch_decode_attention(void*, void*, void*, const void*, const void*,
                             const void*, const void*, const void*, float,
                             int, int, int, int, int, int, int, int,
                             hipStream_t);
void launch_decode_pages(void*, void*, void*, const void*, void*, void*,
                         const void*, const void*, float, int, int, int, int,
                         int, int, int, void*, const DecodeHeads*,
                         hipStream_t);
bool launch_norm_rows(void*, void*, const void*, int, const void*, void*,
                      const void*, float, const void*, int, int, int, int,
                      hipStream_t);
bool launch_stream_rows(void*, void*, int, const void*, const void*, int, int,
                        int, int, hipStream_t);
void launch_place_inputs(void*, const void*, int, void*, const void*, int, int,
                         int, int, hipStream_t);
void launch_prefill_attention(void*, const void*, const void*, const void*,
                              const void*, const void*, float, int, int, int,
                              int, int, int, hipStream_t);
void launch_prefill_flash(void*, const void*, const void*, const void*,
                          const void*, const void*, const void*, float, int,
                          const void*, int, const void*, int, void*, void*, int,
                          int, int, long, long, long, hipStream_t);
void launch_mfma_probe(void*, const void*, const void*, int, int, hipStream_t);
void launch_mfma_probe32(void*, const void*, const void*, int, int, int,
                         hipStream_t);
void launch_kv_peer_copy(void*, const void*, const void*, const void*, int,
                         int, int, long, long, long, long, hipStream_t);
void launch_xgmi_allreduce(void*, const void*, void**, void**, int, int,
                           long, hipStream_t);
long xgmi_allreduce_signal_bytes();
long xgmi_allreduce_error_offset();
long xgmi_allreduce_counter_offset();
}

namespace {

hipStream_t current_stream() {
  return at::hip::getCurrentHIPStream().stream();
}

void check_bf16_contig(const torch::Tensor& t, const char* name) {
  TORCH_CHECK(t.is_cuda(), name, " must be on GPU");
  TORCH_CHECK(t.scalar_type() == torch::kBFloat16, name, " must be bf16");
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
}

torch::Tensor rmsnorm(torch::Tensor x, torch::Tensor weight, double eps) {
  check_bf16_contig(x, "x");
  check_bf16_contig(weight, "weight");
  const int hidden = x.size(-1);
  TORCH_CHECK(hidden % 8 == 0, "hidden must be a multiple of 8");
  const int tokens = x.numel() / hidden;
  auto out = torch::empty_like(x);
  launch_rmsnorm(out.data_ptr(), x.data_ptr(), weight.data_ptr(), (float)eps,
                 tokens, hidden, current_stream());
  return out;
}

void fused_add_rmsnorm(torch::Tensor x, torch::Tensor residual,
                       torch::Tensor weight, double eps) {
  check_bf16_contig(x, "x");
  check_bf16_contig(residual, "residual");
  const int hidden = x.size(-1);
  TORCH_CHECK(hidden % 8 == 0, "hidden must be a multiple of 8");
  const int tokens = x.numel() / hidden;
  launch_fused_add_rmsnorm(x.data_ptr(), residual.data_ptr(),
                           weight.data_ptr(), (float)eps, tokens, hidden,
                           current_stream());
}

// x W^T of a decode batch as its parts' sums, f32 [parts, M, N], for a kernel
// that reads them; bf16 [M, N] where the GEMM is not split.
torch::Tensor skinny_parts(torch::Tensor a, torch::Tensor w) {
  check_skinny(a, w);
  const int64_t M = a.size(0), K = a.size(1), N = w.size(0);
  const SkinnyPlan plan = pick_skinny((int)M, (int)N, (int)K);
  const bool split = plan.splits > 1;
  auto c = split ? torch::empty({plan.splits, M, N},
                                a.options().dtype(torch::kFloat32))
                 : torch::empty({M, N}, a.options());
  launch_skinny_gemm(split ? nullptr : c.data_ptr(),
                     split ? c.data_ptr() : nullptr, a.data_ptr(),
                     w.data_ptr(), (int)M, (int)N, (int)K, plan.waves,
                     plan.splits, 0, current_stream());
  return c;
}

// silu(a Wg^T) * (a Wu^T), w = [Wg; Wu].
torch::Tensor skinny_swiglu(torch::Tensor a, torch::Tensor w) {
  check_skinny(a, w);
  const int64_t M = a.size(0), K = a.size(1), N = w.size(0);
  TORCH_CHECK(M <= 128, "at most 128 rows");
  auto c = torch::empty({M, N / 2}, a.options());
  // as pick_skinny, unsplit; the smaller workgroups where they fill the chip
  const int waves = pick_skinny((int)M, (int)N, (int)K).waves == 0 ? 0
                    : M <= 64 && N <= 16384                        ? 4
                                                                   : 8;
  launch_skinny_gemm(c.data_ptr(), nullptr, a.data_ptr(), w.data_ptr(),
                     (int)M, (int)N, (int)K, waves, 1, 1, current_stream());
  return c;
}

// residual += x (in place); the RMS norm of it.  x: bf16 [T, H], or f32 sums
// [parts, T, H] of skinny_parts.
torch::Tensor add_rmsnorm(torch::Tensor x, torch::Tensor residual,
                          torch::Tensor weight, double eps) {
  const bool split = x.scalar_type() == torch::kFloat32;
  TORCH_CHECK(x.is_cuda() && x.is_contiguous() &&
              (split ? x.dim() == 3 : x.scalar_type() == torch::kBFloat16),
              "x must be bf16 rows or f32 parts of them, contiguous on GPU");
  check_bf16_contig(residual, "residual");
  check_bf16_contig(weight, "weight");
  const int hidden = residual.size(-1);
  const int rows = residual.numel() / hidden;
  TORCH_CHECK(x.size(-1) == hidden && weight.numel() == hidden &&
              x.numel() == (split ? x.size(0) : 1) * residual.numel(),
              "shapes disagree");
  TORCH_CHECK(hidden % 4 == 0 && hidden <= 16384,
              "hidden must be a multiple of 4, at most 16384");
  auto out = torch::empty_like(residual);
  if (rows)
    launch_add_rmsnorm_rows(out.data_ptr(), x.data_ptr(), residual.data_ptr(),
                            weight.data_ptr(), (float)eps,
                            split ? (int)x.size(0) : 0, rows, hidden,
                            current_stream());
  return out;
}

// table's rows of the ids, bf16; below 0 from its end, NaN where there is none
torch::Tensor embed_rows(torch::Tensor ids, torch::Tensor table) {
  check_bf16_contig(table, "table");
  TORCH_CHECK(ids.is_cuda() && ids.is_contiguous() && ids.dim() == 1 &&
              ids.scalar_type() == torch::kInt64, "ids must be int64 on GPU");
  TORCH_CHECK(table.dim() == 2 && table.size(1) % 8 == 0 &&
              (reinterpret_cast<uintptr_t>(table.data_ptr()) & 15) == 0,
              "rows of whole, aligned 16 bytes");
  TORCH_CHECK(table.size(1) > 0 && ids.numel() < (1ll << 31), "sizes");
  auto out = torch::empty({ids.numel(), table.size(1)}, table.options());
  if (ids.numel())
    launch_embed_rows(out.data_ptr(), table.data_ptr(), ids.data_ptr(),
                      table.size(0), (int)table.size(1), (int)ids.numel(),
                      false, current_stream());
  return out;
}

// Is this memory of the host what host_read.h takes it for?
static bool fine_grained(const torch::Tensor& host) {
  unsigned flags = 0;
  if (hipHostGetFlags(&flags, host.data_ptr()) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return !(flags & hipHostMallocNonCoherent);
}

// Pinned memory as a kernel may read it: itself, or its copy on the GPU.
static torch::Tensor for_kernels(const torch::Tensor& host, torch::Device device) {
  return fine_grained(host) ? host : host.to(device, /*non_blocking=*/true);
}

// Memory of the host that a kernel on the current stream has read: torch gives it to
// nobody else before the stream has come so far, if it is of torch's allocator.
static bool held_for_stream(const torch::Tensor& host) {
  const auto stream = at::hip::getCurrentHIPStream();
  return at::getHostAllocator(at::kCUDA)->record_event(
      host.data_ptr(), host.storage().data_ptr().get_context(),
      c10::Stream(c10::Stream::UNSAFE,
                  c10::Device(c10::kCUDA, stream.device_index()), stream.id()));
}

static void read_by_stream(const torch::Tensor& host) {
  if (!held_for_stream(host))
    TORCH_CHECK(hipStreamSynchronize(current_stream()) == hipSuccess,
                "waiting for a read of the host's memory");
}

// Rows of x that the host names, below 0 from its end.
torch::Tensor rows_at(torch::Tensor x, const std::vector<int64_t>& rows) {
  check_bf16_contig(x, "x");
  TORCH_CHECK(x.dim() == 2 && x.size(1) > 0 && x.size(1) % 8 == 0 &&
              (reinterpret_cast<uintptr_t>(x.data_ptr()) & 15) == 0 &&
              rows.size() < (1ull << 31), "rows of whole, aligned 16 bytes");
  const int64_t n = rows.size(), all = x.size(0);
  for (const int64_t r : rows)
    TORCH_CHECK_INDEX(r >= -all && r < all, "row ", r, " of ", all);
  auto out = torch::empty({n, x.size(1)}, x.options());
  if (n == 0) return out;
  auto host = torch::empty({n}, torch::dtype(torch::kInt64).pinned_memory(true));
  std::copy(rows.begin(), rows.end(), host.data_ptr<int64_t>());
  const auto from = for_kernels(host, x.device());
  launch_embed_rows(out.data_ptr(), x.data_ptr(), from.data_ptr(), all,
                    (int)x.size(1), (int)n, true, current_stream());
  read_by_stream(host);
  return out;
}

torch::Tensor silu_mul(torch::Tensor x) {
  if (x.scalar_type() == torch::kFloat32) {     // sums of skinny_parts
    TORCH_CHECK(x.is_cuda() && x.is_contiguous() && x.dim() == 3 &&
                x.size(2) % 8 == 0, "f32 parts [parts, T, 2 I], I % 4 == 0");
    const int64_t tokens = x.size(1), inter = x.size(2) / 2;
    auto out = torch::empty({tokens, inter},
                            x.options().dtype(torch::kBFloat16));
    if (tokens)
      launch_silu_parts(out.data_ptr(), x.data_ptr(), (int)x.size(0),
                        (int)tokens, (int)inter, current_stream());
    return out;
  }
  check_bf16_contig(x, "x");
  const int inter2 = x.size(-1);
  TORCH_CHECK(inter2 % 16 == 0, "2*inter must be a multiple of 16");
  const int inter = inter2 / 2;
  const int tokens = x.numel() / inter2;
  auto out = torch::empty({x.size(0), inter}, x.options());
  launch_silu_mul(out.data_ptr(), x.data_ptr(), tokens, inter,
                  current_stream());
  return out;
}

static void check_bf16_rowslice(const torch::Tensor& t, const char* name) {
  // bf16 on GPU, [T, W] or [T, H, D], innermost dims contiguous; the
  // TOKEN stride may be wider (a column slice of the fused QKV buffer)
  TORCH_CHECK(t.is_cuda(), name, " must be on GPU");
  TORCH_CHECK(t.scalar_type() == torch::kBFloat16, name, " must be bf16");
  if (t.dim() == 2) {
    TORCH_CHECK(t.stride(1) == 1, name, " rows must be contiguous");
  } else {
    TORCH_CHECK(t.dim() == 3 && t.stride(2) == 1 &&
                t.stride(1) == t.size(2), name,
                " must be [T, H, D] with contiguous (H, D) rows");
  }
}

void rope_store_kv(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                   torch::Tensor key_cache, torch::Tensor value_cache,
                   torch::Tensor cos_sin, torch::Tensor positions,
                   torch::Tensor slot_mapping) {
  check_bf16_rowslice(q, "q");
  check_bf16_rowslice(k, "k");
  check_bf16_rowslice(v, "v");
  TORCH_CHECK(k.stride(0) == v.stride(0), "k/v stride mismatch");
  TORCH_CHECK(cos_sin.scalar_type() == torch::kFloat32, "cos_sin fp32");
  TORCH_CHECK(positions.scalar_type() == torch::kInt32, "positions int32");
  TORCH_CHECK(slot_mapping.scalar_type() == torch::kInt32, "slots int32");
  const int tokens = q.size(0);
  const int head_dim = key_cache.size(3);
  const int num_kv_heads = key_cache.size(1);
  const int page_size = key_cache.size(2);
  const int num_q_heads = (int)(q.numel() / tokens / head_dim);
  const auto aligned = [](const torch::Tensor& t) {
    return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
  };
  // 16-byte accesses need rows that begin at multiples of them (32 + 8 heads,
  // 1 / 2048 tokens: 3.9 / 12.3 us of the kernel for any size against 2.3 / 8.7)
  if (head_dim == 128 && q.stride(0) % 8 == 0 && k.stride(0) % 8 == 0 &&
      aligned(q) && aligned(k) && aligned(v) && aligned(key_cache) &&
      aligned(value_cache) && aligned(cos_sin)) {
    launch_rope_heads(q.data_ptr(), k.data_ptr(), v.data_ptr(), nullptr, 0,
                      nullptr, nullptr, 0.f, key_cache.data_ptr(),
                      value_cache.data_ptr(), cos_sin.data_ptr(),
                      positions.data_ptr(), slot_mapping.data_ptr(), tokens,
                      num_q_heads, num_kv_heads, page_size,
                      (int)q.stride(0), (int)k.stride(0), current_stream());
    return;
  }
  launch_rope_store_kv(q.data_ptr(), k.data_ptr(), v.data_ptr(),
                       key_cache.data_ptr(), value_cache.data_ptr(),
                       cos_sin.data_ptr(), positions.data_ptr(),
                       slot_mapping.data_ptr(), tokens, num_q_heads,
                       num_kv_heads, head_dim, page_size,
                       (int)q.stride(0), (int)k.stride(0),
                       current_stream());
}

// Norm of the query and key heads (optional), rotation and paged store of a
// fused projection: bf16 [T, width], changed in place, or f32 sums [parts, T,
// width] of skinny_parts.  Returns the projection in bf16.
torch::Tensor rope_heads(torch::Tensor proj, int64_t num_q_heads,
                         c10::optional<torch::Tensor> q_norm,
                         c10::optional<torch::Tensor> k_norm, double eps,
                         torch::Tensor key_cache, torch::Tensor value_cache,
                         torch::Tensor cos_sin, torch::Tensor positions,
                         torch::Tensor slot_mapping) {
  const bool split = proj.scalar_type() == torch::kFloat32;
  TORCH_CHECK(proj.is_cuda() && proj.is_contiguous() &&
              (split ? proj.dim() == 3
                     : proj.dim() == 2 &&
                           proj.scalar_type() == torch::kBFloat16),
              "projection must be bf16 rows or f32 parts of them");
  check_bf16_contig(key_cache, "key_cache");
  check_bf16_contig(value_cache, "value_cache");
  TORCH_CHECK(cos_sin.scalar_type() == torch::kFloat32 &&
              cos_sin.is_contiguous() && cos_sin.size(1) == 128,
              "cos_sin must be fp32 [positions, 128]");
  TORCH_CHECK(positions.scalar_type() == torch::kInt32 &&
              slot_mapping.scalar_type() == torch::kInt32,
              "positions and slots int32");
  const int64_t tokens = proj.size(-2), width = proj.size(-1);
  const int64_t kv_heads = key_cache.size(1);
  TORCH_CHECK(key_cache.size(3) == 128 &&
              width == (num_q_heads + 2 * kv_heads) * 128,
              "heads of 128, q | k | v");
  TORCH_CHECK(positions.numel() == tokens && slot_mapping.numel() == tokens,
              "a position and a slot per token");
  TORCH_CHECK(q_norm.has_value() == k_norm.has_value(), "both norms or none");
  for (const auto& n : {q_norm, k_norm})
    if (n.has_value()) {
      check_bf16_contig(*n, "norm");
      TORCH_CHECK(n->numel() == 128, "norms of 128");
    }
  TORCH_CHECK(tokens * (width / 128) < (1ll << 31) - 32, "too many rows");
  auto out = split ? torch::empty({tokens, width},
                                  proj.options().dtype(torch::kBFloat16))
                   : proj;
  if (tokens == 0) return out;
  auto* base = static_cast<uint16_t*>(out.data_ptr());
  launch_rope_heads(base, base + num_q_heads * 128,
                    base + (num_q_heads + kv_heads) * 128,
                    split ? proj.data_ptr() : nullptr,
                    split ? (int)proj.size(0) : 0,
                    q_norm ? q_norm->data_ptr() : nullptr,
                    k_norm ? k_norm->data_ptr() : nullptr, (float)eps,
                    key_cache.data_ptr(), value_cache.data_ptr(),
                    cos_sin.data_ptr(), positions.data_ptr(),
                    slot_mapping.data_ptr(), (int)tokens, (int)num_q_heads,
                    (int)kv_heads, (int)key_cache.size(2), (int)width,
                    (int)width, current_stream());
  return out;
}

// silu(a Wg^T) * (a Wu^T) of up to 4 rows, w = [Wg; Wu]
torch::Tensor stream_swiglu(torch::Tensor a, torch::Tensor w) {
  check_skinny(a, w);
  const int64_t M = a.size(0), K = a.size(1), N = w.size(0);
  auto c = torch::empty({M, N / 2}, a.options());
  TORCH_CHECK(launch_stream_rows(c.data_ptr(), nullptr, 0, a.data_ptr(),
                                 w.data_ptr(), (int)M, (int)N, (int)K, 1,
                                 current_stream()),
              "at most 4 rows");
  return c;
}

// Up to 4 rows: the RMS norm of residual + src (bf16, or f32 sums [1, M, K] of
// stream_linear; it may be missing), a GEMM and its end in one launch: the product in
// bf16 (0, which the models leave for 2), silu(gate) * up (1; what launch_norm_rows
// refuses behind a launch of the norm's own, which ops.norm_swiglu does in place), or
// the product's f32 sums [1, M, N] (2).  Returns that and the new residual, which is
// another tensor unless src is missing.
std::vector<torch::Tensor> norm_rows(c10::optional<torch::Tensor> src,
                                     torch::Tensor residual,
                                     torch::Tensor norm_weight, double eps,
                                     torch::Tensor w, int64_t end) {
  check_skinny(residual, w);
  check_bf16_contig(norm_weight, "norm weight");
  const int64_t M = residual.size(0), K = residual.size(1), N = w.size(0);
  TORCH_CHECK(norm_weight.numel() == K, "norm weight of K");
  TORCH_CHECK(end >= 0 && end <= 2, "unknown end");
  const bool sums = src && src->scalar_type() == torch::kFloat32;
  if (src) {
    TORCH_CHECK(src->is_cuda() && src->is_contiguous() &&
                src->numel() == residual.numel() && src->size(-1) == K &&
                (sums || src->scalar_type() == torch::kBFloat16),
                "src like residual, or f32 sums");
  }
  if (end == 1 && M > 1 && (sums || (M > 2 && K > 4096))) {
    auto next = src ? residual.clone() : residual;
    return {stream_swiglu(src ? add_rmsnorm(*src, next, norm_weight, eps)
                              : rmsnorm(residual, norm_weight, eps), w),
            next};
  }
  const auto f32 = residual.options().dtype(torch::kFloat32);
  auto out = end == 2 ? torch::empty({1, M, N}, f32)
                      : torch::empty({M, end == 1 ? N / 2 : N},
                                     residual.options());
  auto next = src ? torch::empty_like(residual) : residual;
  TORCH_CHECK(launch_norm_rows(end == 2 ? nullptr : out.data_ptr(),
                               end == 2 ? out.data_ptr() : nullptr,
                               src ? src->data_ptr() : nullptr, sums,
                               residual.data_ptr(), next.data_ptr(),
                               norm_weight.data_ptr(), (float)eps, w.data_ptr(),
                               (int)M, (int)N, (int)K, end == 1,
                               current_stream()),
              "at most 4 rows of 1024 to 8192");
  return {out, next};
}

// a W^T of up to 4 rows, in bf16 (0), in bf16's values as f32 (1), or its f32 sums as
// one part [1, M, N] (2)
torch::Tensor stream_linear(torch::Tensor a, torch::Tensor w, int64_t end) {
  check_skinny(a, w);
  const int64_t M = a.size(0), K = a.size(1), N = w.size(0);
  TORCH_CHECK(end >= 0 && end <= 2, "unknown end");
  auto c = torch::empty({M, N}, end ? a.options().dtype(torch::kFloat32)
                                    : a.options());
  TORCH_CHECK(launch_stream_rows(end ? nullptr : c.data_ptr(),
                                 end ? c.data_ptr() : nullptr, end == 1,
                                 a.data_ptr(), w.data_ptr(), (int)M, (int)N,
                                 (int)K, 0, current_stream()),
              "at most 4 rows");
  return end == 2 ? c.unsqueeze(0) : c;
}

// fields and tables [rows, width]: a captured step's inputs, from new ones of the host,
// whose tables are [seqs, used].  The kernel reads pinned memory, whose pages the GPU
// maps.
void place_host_inputs(torch::Tensor fields, torch::Tensor tables,
                       torch::Tensor new_fields, torch::Tensor new_tables) {
  for (const auto& t : {fields, new_fields})
    TORCH_CHECK(t.is_contiguous() && t.scalar_type() == torch::kInt64,
                "fields: int64");
  for (const auto& t : {tables, new_tables})
    TORCH_CHECK(t.is_contiguous() && t.dim() == 2 &&
                t.scalar_type() == torch::kInt32, "tables: int32");
  TORCH_CHECK(fields.is_cuda() && tables.is_cuda() && new_fields.is_cpu() &&
              new_tables.is_cpu(), "inputs on GPU, new ones on the host");
  TORCH_CHECK(fields.numel() == new_fields.numel() &&
              new_tables.size(0) <= tables.size(0) &&
              new_tables.size(1) <= tables.size(1), "sizes disagree");
  TORCH_CHECK(fields.numel() < (1 << 30) && tables.numel() < (1 << 30),
              "too many");
  const size_t head = new_fields.nbytes(), rest = new_tables.nbytes();
  if (head + rest == 0 && tables.numel() == 0) return;
  auto host = torch::empty({(int64_t)std::max<size_t>(head + rest, 16)},
                           torch::dtype(torch::kUInt8).pinned_memory(true));
  char* at = (char*)host.data_ptr();
  if (head) std::memcpy(at, new_fields.data_ptr(), head);
  if (rest) std::memcpy(at + head, new_tables.data_ptr(), rest);
  const auto from = for_kernels(host, fields.device());
  at = (char*)from.data_ptr();
  launch_place_inputs(fields.data_ptr(), at, (int)fields.numel(),
                      tables.data_ptr(), at + head, (int)tables.size(0),
                      (int)tables.size(1), (int)new_tables.size(0),
                      (int)new_tables.size(1), current_stream());
  read_by_stream(host);
}

// span: of form 7, the fewest keys that a part has, where the sequence is longer.
// tickets: of form 7 on pages of 16, zeros for every sequence and key head, which
// they are again afterwards: the sequences' last workgroups add up the parts.
torch::Tensor decode_attention(torch::Tensor q, torch::Tensor key_cache,
                               torch::Tensor value_cache,
                               torch::Tensor block_tables,
                               torch::Tensor context_lens, double scale,
                               int64_t num_splits, int64_t wide,
                               int64_t span,
                               c10::optional<torch::Tensor> tickets) {
  // q may be a slice of the fused QKV projection: 3-D bf16 with
  // contiguous (head, dim) rows and an arbitrary token stride
  TORCH_CHECK(q.is_cuda() && q.scalar_type() == torch::kBFloat16 &&
              q.dim() == 3 && q.stride(2) == 1 &&
              q.stride(1) == q.size(2), "q must be [T, QH, D] row-sliced");
  const int num_seqs = q.size(0);
  const int num_q_heads = q.size(1);
  const int head_dim = q.size(2);
  TORCH_CHECK(head_dim == 128, "head_dim must be 128");
  const int num_kv_heads = key_cache.size(1);
  const int page_size = key_cache.size(2);
  const int max_pages = block_tables.size(1);
  const int qpg = num_q_heads / num_kv_heads;
  TORCH_CHECK(qpg == 1 || qpg == 2 || qpg == 4 || qpg == 8,
              "GQA group must be 1/2/4/8");
  TORCH_CHECK(block_tables.scalar_type() == torch::kInt32, "tables int32");
  TORCH_CHECK(context_lens.scalar_type() == torch::kInt32, "lens int32");
  auto out = torch::empty({num_seqs, num_q_heads, head_dim}, q.options());
  torch::Tensor partial_o, partial_ml;
  void *po = nullptr, *pml = nullptr;
  if (num_splits > 1) {
    auto opts = q.options().dtype(torch::kFloat32);
    partial_o = torch::empty({num_splits, num_seqs, num_q_heads, head_dim}, opts);
    partial_ml = torch::empty({num_splits, num_seqs, num_q_heads, 2}, opts);
    po = partial_o.data_ptr();
    pml = partial_ml.data_ptr();
  }
  if (tickets)
    TORCH_CHECK(tickets->is_cuda() && tickets->is_contiguous() &&
                tickets->scalar_type() == torch::kInt32 &&
                tickets->numel() >= (int64_t)num_seqs * num_kv_heads,
                "an int32 ticket per sequence and key head");
  if (wide == 7 && page_size == 16) {
    launch_decode_pages(out.data_ptr(), po, pml, q.data_ptr(),
                        key_cache.data_ptr(), value_cache.data_ptr(),
                        block_tables.data_ptr(), context_lens.data_ptr(),
                        (float)scale, num_seqs, num_q_heads, num_kv_heads,
                        max_pages, (int)num_splits, (int)span,
                        (int)q.stride(0),
                        tickets ? tickets->data_ptr() : nullptr, nullptr,
                        current_stream());
    return out;
  }
  launch_decode_attention(out.data_ptr(), po, pml, q.data_ptr(),
                          key_cache.data_ptr(), value_cache.data_ptr(),
                          block_tables.data_ptr(), context_lens.data_ptr(),
                          (float)scale, num_seqs, num_q_heads, num_kv_heads,
                          page_size, max_pages, (int)num_splits, (int)wide,
                          (int)q.stride(0), current_stream());
  return out;
}

// rope_heads of one row a sequence and decode_attention by form 7 on pages of 16,
// in one launch.  lens count the new token, whose slot no other sequence reads.
torch::Tensor decode_heads(torch::Tensor proj, int64_t heads,
                           c10::optional<torch::Tensor> q_norm,
                           c10::optional<torch::Tensor> k_norm, double eps,
                           torch::Tensor key_cache, torch::Tensor value_cache,
                           torch::Tensor cos_sin, torch::Tensor positions,
                           torch::Tensor slots, torch::Tensor block_tables,
                           torch::Tensor lens, double scale, int64_t splits,
                           int64_t span,
                           c10::optional<torch::Tensor> tickets) {
  const bool parted = proj.scalar_type() == torch::kFloat32;
  TORCH_CHECK(proj.is_cuda() && proj.is_contiguous() &&
              (parted ? proj.dim() == 3 && proj.size(0) >= 1
                      : proj.dim() == 2 &&
                            proj.scalar_type() == torch::kBFloat16),
              "projection must be bf16 rows or f32 parts of them");
  check_bf16_contig(key_cache, "key_cache");
  check_bf16_contig(value_cache, "value_cache");
  const int64_t seqs = proj.size(-2), width = proj.size(-1);
  const int64_t kv_heads = key_cache.size(1), pages = block_tables.size(1);
  TORCH_CHECK(key_cache.dim() == 4 && key_cache.size(2) == 16 &&
              key_cache.size(3) == 128 && key_cache.size(0) >= 1 &&
              value_cache.sizes() == key_cache.sizes(),
              "pages of 16 keys of 128");
  TORCH_CHECK(kv_heads >= 1 && width == (heads + 2 * kv_heads) * 128 &&
              heads % kv_heads == 0, "heads of 128, q | k | v");
  const int64_t group = heads / kv_heads;
  TORCH_CHECK(group == 1 || group == 2 || group == 4 || group == 8,
              "GQA group must be 1/2/4/8");
  TORCH_CHECK(cos_sin.is_cuda() && cos_sin.scalar_type() == torch::kFloat32 &&
              cos_sin.is_contiguous() && cos_sin.dim() == 2 &&
              cos_sin.size(1) == 128, "cos_sin must be fp32 [positions, 128]");
  for (const auto& t : {positions, slots, lens})
    TORCH_CHECK(t.is_cuda() && t.is_contiguous() &&
                t.scalar_type() == torch::kInt32, "an int32 per sequence");
  // lengths and tables may be those of a larger batch, as decode_attention takes them
  TORCH_CHECK(positions.numel() == seqs && slots.numel() == seqs &&
              lens.numel() >= seqs, "a position, slot and length per sequence");
  TORCH_CHECK(block_tables.is_cuda() && block_tables.is_contiguous() &&
              block_tables.dim() == 2 && block_tables.size(0) >= seqs &&
              pages >= 1 && block_tables.scalar_type() == torch::kInt32,
              "int32 page tables");
  TORCH_CHECK(q_norm.has_value() == k_norm.has_value(), "both norms or none");
  for (const auto& n : {q_norm, k_norm})
    if (n.has_value()) {
      check_bf16_contig(*n, "norm");
      TORCH_CHECK(n->numel() == 128, "norms of 128");
    }
  TORCH_CHECK(splits >= 1 && splits < 65536 && seqs < 65536 && span >= 1 &&
              seqs * width < (1ll << 31), "parts");
  if (tickets)
    TORCH_CHECK(tickets->is_cuda() && tickets->is_contiguous() &&
                tickets->scalar_type() == torch::kInt32 &&
                tickets->numel() >= seqs * kv_heads,
                "an int32 ticket per sequence and key head");
  auto opts = proj.options().dtype(torch::kFloat32);
  auto out = torch::empty({seqs, heads, 128},
                          proj.options().dtype(torch::kBFloat16));
  if (seqs == 0) return out;
  torch::Tensor sums;           // of every part, then maximum and sum of each row
  float *po = nullptr, *pml = nullptr;
  if (splits > 1) {
    const int64_t rows = splits * seqs * heads;
    sums = torch::empty({rows * 130}, opts);
    po = sums.data_ptr<float>();
    pml = po + rows * 128;
  }
  const auto norm = [](const c10::optional<torch::Tensor>& t) -> const void* {
    return t ? t->data_ptr() : nullptr;
  };
  const DecodeHeads in{parted ? proj.data_ptr<float>() : nullptr,
                       positions.data_ptr<int>(), slots.data_ptr<int>(),
                       cos_sin.data_ptr<float>(), norm(q_norm), norm(k_norm),
                       (float)eps, parted ? (int)proj.size(0) : 0};
  launch_decode_pages(out.data_ptr(), po, pml,
                      parted ? nullptr : proj.data_ptr(),
                      key_cache.data_ptr(), value_cache.data_ptr(),
                      block_tables.data_ptr(), lens.data_ptr(), (float)scale,
                      (int)seqs, (int)heads, (int)kv_heads, (int)pages,
                      (int)splits, (int)span, (int)width,
                      tickets ? tickets->data_ptr() : nullptr, &in,
                      current_stream());
  return out;
}

// Blocks, lengths, items, joins and parts of prompt attention (PrefillPlan), by one
// copy from pinned memory, which torch keeps until the copy is done.
std::tuple<torch::Tensor, torch::Tensor, c10::optional<torch::Tensor>,
           c10::optional<torch::Tensor>, int64_t>
prefill_plan(const std::vector<int64_t>& cu, const std::vector<int64_t>& cu_k,
             int64_t heads, int64_t kv_heads, torch::Device device) {
  TORCH_CHECK(cu.size() >= 1 && cu.size() == cu_k.size() && kv_heads >= 1 &&
              heads >= kv_heads, "where query and key rows begin, and heads");
  const int64_t tokens = 128 / (heads / kv_heads);
  for (size_t i = 1; i < cu.size(); ++i)
    TORCH_CHECK(cu[i] - cu[i - 1] > -std::max<int64_t>(tokens, 1), "rows before those of the last");
  const PrefillWork work = plan_prefill(cu, cu_k, tokens, kv_heads);
  const std::vector<int32_t>* arrays[] = {&work.blocks, &work.lens, &work.items,
                                          &work.joins};
  int64_t begin[4], total = 0;
  for (int i = 0; i < 4; ++i) {         // each at a multiple of 16 bytes
    begin[i] = total;
    total += ((int64_t)arrays[i]->size() + 3) / 4 * 4;
  }
  const auto opts = torch::dtype(torch::kInt32);
  auto host = torch::empty({std::max<int64_t>(total, 4)},
                           opts.pinned_memory(device.is_cuda()));
  for (int i = 0; i < 4; ++i)
    std::copy(arrays[i]->begin(), arrays[i]->end(),
              host.data_ptr<int32_t>() + begin[i]);
  auto all = host.to(device, /*non_blocking=*/true);
  const auto part = [&](int i, int64_t width) {
    const int64_t n = arrays[i]->size() / width;
    return width == 1 ? all.as_strided({n}, {1}, begin[i])
                      : all.as_strided({n, width}, {width, 1}, begin[i]);
  };
  c10::optional<torch::Tensor> items, joins;
  if (work.parts) {
    items = part(2, 4);
    joins = part(3, 3);
  }
  return {part(0, 4), part(1, 1), items, joins, work.parts};
}

torch::Tensor prefill_attention(torch::Tensor q, torch::Tensor k,
                                torch::Tensor v, torch::Tensor block_info,
                                torch::Tensor seq_lens, double scale,
                                int64_t swz) {
  auto rowsliced3 = [](const torch::Tensor& t, const char* name) {
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kBFloat16 &&
                t.dim() == 3 && t.stride(2) == 1 &&
                t.stride(1) == t.size(2), name,
                " must be [T, H, D] row-sliced");
  };
  rowsliced3(q, "q");
  rowsliced3(k, "k");
  rowsliced3(v, "v");
  TORCH_CHECK(k.stride(0) == v.stride(0), "k/v stride mismatch");
  TORCH_CHECK(q.size(2) == 128, "head_dim must be 128");
  TORCH_CHECK(block_info.scalar_type() == torch::kInt32, "block_info int32");
  TORCH_CHECK(seq_lens.scalar_type() == torch::kInt32, "seq_lens int32");
  const int nblocks = block_info.size(0);
  const int num_q_heads = q.size(1);
  const int num_kv_heads = k.size(1);
  auto out = torch::empty({q.size(0), (int64_t)num_q_heads, (int64_t)128},
                          q.options());
  launch_prefill_attention(out.data_ptr(), q.data_ptr(), k.data_ptr(),
                           v.data_ptr(), block_info.data_ptr(),
                           seq_lens.data_ptr(), (float)scale, nblocks,
                           num_q_heads, num_kv_heads, (int)swz,
                           (int)q.stride(0), (int)k.stride(0),
                           current_stream());
  return out;
}

// Causal attention of prompt rows.  k and v are rows [Tkv, H, 128], or, with
// slots [Tkv], pages [pages, H, page_size, 128] that the slots name rows of.
// block_info [n, 4] and seq_lens [n]: a workgroup's first query row of the
// sequence, its number among the sequence's blocks of 128 / (QH / H) tokens,
// the sequence's first kv row and the position of its first query row; its kv
// rows.  items [m, 4] and joins [c, 3], where work is cut by keys: a
// workgroup's block, its first and one past its last tile of 64 keys, and the
// part that its sums are, or -1 for all of a block; a cut block, its first part
// and how many they are, in order of the parts.
torch::Tensor prefill_flash(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                            torch::Tensor block_info, torch::Tensor seq_lens,
                            double scale, c10::optional<torch::Tensor> slots,
                            c10::optional<torch::Tensor> items,
                            c10::optional<torch::Tensor> joins,
                            int64_t parts) {
  auto rows3 = [](const torch::Tensor& t, const char* name) {
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kBFloat16 &&
                t.dim() == 3 && t.stride(2) == 1 &&
                t.stride(1) == t.size(2) && t.size(2) == 128, name,
                " must be [T, H, 128] row-sliced");
  };
  rows3(q, "q");
  // the kernel brings pieces of 16 bytes to LDS
  if ((reinterpret_cast<uintptr_t>(q.data_ptr()) | q.stride(0) * 2) & 15)
    q = q.clone(at::MemoryFormat::Contiguous);
  int shift = 0;
  if (slots.has_value()) {
    check_bf16_contig(k, "keys");
    check_bf16_contig(v, "values");
    TORCH_CHECK(k.dim() == 4 && k.sizes() == v.sizes() && k.size(3) == 128,
                "pages must be [pages, H, page_size, 128]");
    while ((1 << shift) < k.size(2)) ++shift;
    TORCH_CHECK((1 << shift) == k.size(2), "page size: a power of 2");
    TORCH_CHECK(slots->is_cuda() && slots->is_contiguous() &&
                slots->scalar_type() == torch::kInt32, "slots int32");
  } else {
    rows3(k, "k");
    rows3(v, "v");
    TORCH_CHECK(k.stride(0) == v.stride(0), "k/v stride mismatch");
  }
  for (const auto& t : {block_info, seq_lens})
    TORCH_CHECK(t.is_cuda() && t.is_contiguous() &&
                t.scalar_type() == torch::kInt32, "plan int32");
  const int blocks = seq_lens.numel();
  TORCH_CHECK(block_info.numel() == 4 * (int64_t)blocks, "plan sizes");
  const int heads = q.size(1), kv_heads = k.size(1);
  TORCH_CHECK(kv_heads > 0 && heads % kv_heads == 0 && heads / kv_heads <= 128,
              "query heads: a multiple of the key heads, at most 128 times");
  TORCH_CHECK(items.has_value() == joins.has_value(), "items and joins");
  if (items)
    for (const auto& t : {*items, *joins})
      TORCH_CHECK(t.is_cuda() && t.is_contiguous() && t.dim() == 2 &&
                  t.scalar_type() == torch::kInt32, "plan int32");
  TORCH_CHECK(!items || (items->size(1) == 4 && joins->size(1) == 3 &&
                         parts >= 0), "plan sizes");
  auto out = torch::empty({q.size(0), (int64_t)heads, (int64_t)128},
                          q.options());
  torch::Tensor sums;           // per part and key head 128 rows of 128, then
  float* ml = nullptr;          // maximum and sum of each row
  if (items && parts > 0) {
    const int64_t rows = parts * kv_heads * 128;
    sums = torch::empty({rows * 130}, q.options().dtype(torch::kFloat32));
    ml = sums.data_ptr<float>() + rows * 128;
  }
  launch_prefill_flash(out.data_ptr(), q.data_ptr(), k.data_ptr(),
                       v.data_ptr(), slots ? slots->data_ptr() : nullptr,
                       block_info.data_ptr(), seq_lens.data_ptr(),
                       (float)scale, blocks,
                       items ? items->data_ptr() : nullptr,
                       items ? (int)items->size(0) : 0,
                       items ? joins->data_ptr() : nullptr,
                       items ? (int)joins->size(0) : 0,
                       ml ? sums.data_ptr() : nullptr, ml, heads, kv_heads,
                       shift, q.stride(0), k.stride(0),
                       slots ? k.size(0) * k.size(1) * k.size(2) : 0,
                       current_stream());
  return out;
}

// Who takes a product of many rows (ops.block_routes).
enum Route { BY_LIBRARY, BY_SKINNY, BY_TILE, GLU_BY_SKINNY, GLU_BY_TILE };

static torch::Tensor routed(const torch::Tensor& x, const torch::Tensor& w,
                            int64_t route) {
  switch (route) {
    case BY_SKINNY: return skinny_parts(x, w);
    case BY_TILE: return tile_parts(x, w);
    case GLU_BY_SKINNY: return skinny_swiglu(x, w);
    case GLU_BY_TILE: return tile_swiglu(x, w);
    default: return at::linear(x, w);
  }
}

// ops.add_rmsnorm, or the norm of the residual alone
static torch::Tensor prompt_norm(const c10::optional<torch::Tensor>& src,
                                 const torch::Tensor& residual,
                                 const torch::Tensor& weight, double eps) {
  if (!src) return rmsnorm(residual, weight, eps);
  if (src->scalar_type() == torch::kFloat32 ||
      (src->size(0) <= 256 && src->size(-1) <= 16384))
    return add_rmsnorm(*src, residual, weight, eps);
  fused_add_rmsnorm(*src, residual, weight, eps);
  return *src;
}

// Rows that the blocks below take.  Up to four take norm and product in one
// launch, by norm_rows.
static bool block_rows(const torch::Tensor& residual) {
  return residual.is_cuda() && residual.dim() == 2 && residual.size(0) > 4 &&
         residual.size(1) % 8 == 0 && !at::GradMode::is_enabled();
}

// Weights that not only the library takes.
static bool block_weight(const torch::Tensor& w) {
  return w.is_cuda() && w.is_contiguous() && w.dim() == 2 &&
         w.scalar_type() == torch::kBFloat16 &&
         (reinterpret_cast<uintptr_t>(w.data_ptr()) & 15) == 0;
}

// The two blocks of a Llama layer on many rows: the launches of their operations
// (models/llama.py), issued by one call each.  Short prompts wait for the host: 37
// tokens of 2048 wide are 61 launches in six layers, whose kernels take 400 us and
// which take 600 to issue, 478 so; a step among others takes 442.  (A whole layer
// by one call 425, but hooked, replaced or substituted parts of it were passed by.)
// Routes: of the products with the two weights.  Both return the block's result
// for the next norm to add, and add to the residual in place; none, and nothing
// is done, for what only the operations by themselves take.
c10::optional<torch::Tensor> prompt_attention_block(
    c10::optional<torch::Tensor> src, torch::Tensor residual,
    torch::Tensor norm, double eps, torch::Tensor wqkv, torch::Tensor wo,
    std::pair<int64_t, int64_t> routes, int64_t heads,
    c10::optional<torch::Tensor> q_norm, c10::optional<torch::Tensor> k_norm,
    torch::Tensor key_cache, torch::Tensor value_cache, torch::Tensor cos_sin,
    torch::Tensor positions, torch::Tensor slot_mapping, double scale,
    torch::Tensor block_info, torch::Tensor seq_lens,
    c10::optional<torch::Tensor> items, c10::optional<torch::Tensor> joins,
    int64_t parts, c10::optional<torch::Tensor> gather_slots) {
  const int64_t rows = residual.size(0), kvh = key_cache.size(1);
  const int64_t page = key_cache.size(2);
  if (!block_rows(residual) || !block_weight(wqkv) || !block_weight(wo) ||
      key_cache.size(3) != 128 || heads % kvh || heads / kvh > 128 ||
      (gather_slots && (page & (page - 1))))
    return c10::nullopt;
  auto qkv = rope_heads(
      routed(prompt_norm(src, residual, norm, eps), wqkv, routes.first), heads,
      q_norm, k_norm, eps, key_cache, value_cache, cos_sin, positions,
      slot_mapping);
  const auto part = [&](int64_t from, int64_t n) {
    return qkv.narrow(1, from * 128, n * 128).view({rows, n, 128});
  };
  // behind a past: all rows, the new ones too, from the pages
  auto o = prefill_flash(part(0, heads),
                         gather_slots ? key_cache : part(heads, kvh),
                         gather_slots ? value_cache : part(heads + kvh, kvh),
                         block_info, seq_lens, scale, gather_slots, items,
                         joins, parts);
  return routed(o.view({rows, heads * 128}), wo, routes.second);
}

c10::optional<torch::Tensor> swiglu_block(
    c10::optional<torch::Tensor> src, torch::Tensor residual,
    torch::Tensor norm, double eps, torch::Tensor w_gate_up,
    torch::Tensor w_down, std::pair<int64_t, int64_t> routes) {
  if (!block_rows(residual) || !block_weight(w_gate_up) ||
      !block_weight(w_down))
    return c10::nullopt;
  auto x = routed(prompt_norm(src, residual, norm, eps), w_gate_up,
                  routes.first);
  if (routes.first != GLU_BY_SKINNY && routes.first != GLU_BY_TILE)
    x = silu_mul(x);
  return routed(x, w_down, routes.second);
}

torch::Tensor mfma_probe(torch::Tensor a, torch::Tensor b, int64_t a_split,
                         int64_t b_split) {
  auto d = torch::zeros({16, 16}, a.options().dtype(torch::kFloat32));
  launch_mfma_probe(d.data_ptr(), a.data_ptr(), b.data_ptr(), (int)a_split,
                    (int)b_split, current_stream());
  return d;
}

torch::Tensor mfma_probe32(torch::Tensor a, torch::Tensor b, int64_t a_split,
                           int64_t b_split, int64_t dmap) {
  auto d = torch::zeros({32, 32}, a.options().dtype(torch::kFloat32));
  launch_mfma_probe32(d.data_ptr(), a.data_ptr(), b.data_ptr(), (int)a_split,
                      (int)b_split, (int)dmap, current_stream());
  return d;
}

}  // namespace

// ---- KV-pool IPC export + xGMI peer push (parallel/kv_peer.py) -----------
// The decode engine's KV pool is allocated with hipMalloc directly (not the
// caching allocator) so data_ptr() IS the allocation base hipIpcGetMemHandle
// requires; the prefill process maps it with lazy peer access (the xGMI
// route) and pushes pages with the kv_peer_copy kernel.

torch::Tensor ipc_alloc_bf16(std::vector<int64_t> sizes) {
  int64_t numel = 1;
  for (auto s : sizes) numel *= s;
  void* ptr = nullptr;
  hipError_t err = hipMalloc(&ptr, numel * 2);
  TORCH_CHECK(err == hipSuccess, "hipMalloc(", numel * 2,
              " B) failed: ", hipGetErrorString(err));
  int dev = 0;
  (void)hipGetDevice(&dev);
  auto opts = torch::TensorOptions()
                  .dtype(torch::kBFloat16)
                  .device(torch::kCUDA, dev);
  return torch::from_blob(
      ptr, sizes, [](void* p) { (void)hipFree(p); }, opts);
}

py::bytes kv_ipc_export(torch::Tensor pool) {
  TORCH_CHECK(pool.is_cuda(), "pool must be on GPU");
  hipIpcMemHandle_t handle;
  hipError_t err = hipIpcGetMemHandle(&handle, pool.data_ptr());
  TORCH_CHECK(err == hipSuccess,
              "hipIpcGetMemHandle failed (pool must be an ipc_alloc_bf16 "
              "base allocation): ", hipGetErrorString(err));
  return py::bytes(reinterpret_cast<const char*>(&handle), sizeof(handle));
}

int64_t kv_ipc_open(std::string raw) {
  // std::string parameter: converted from py::bytes during argument
  // processing (GIL held) so the gil_scoped_release guard is safe
  TORCH_CHECK(raw.size() == sizeof(hipIpcMemHandle_t), "bad handle size");
  hipIpcMemHandle_t handle;
  memcpy(&handle, raw.data(), sizeof(handle));
  void* ptr = nullptr;
  hipError_t err =
      hipIpcOpenMemHandle(&ptr, handle, hipIpcMemLazyEnablePeerAccess);
  TORCH_CHECK(err == hipSuccess,
              "hipIpcOpenMemHandle failed: ", hipGetErrorString(err));
  return reinterpret_cast<int64_t>(ptr);
}

void kv_ipc_close(int64_t ptr) {
  hipError_t err = hipIpcCloseMemHandle(reinterpret_cast<void*>(ptr));
  TORCH_CHECK(err == hipSuccess,
              "hipIpcCloseMemHandle failed: ", hipGetErrorString(err));
}

void kv_peer_copy(int64_t dst_base, torch::Tensor src_kv,
                  torch::Tensor src_pages, torch::Tensor dst_pages,
                  int64_t dst_num_pages) {
  // src_kv: [L, 2, Ps, kvh, ps, hd] bf16 contiguous; dst pool has the SAME
  // per-page layout but its own page count (dst_num_pages)
  check_bf16_contig(src_kv, "src_kv");
  TORCH_CHECK(src_kv.dim() == 6 && src_kv.size(1) == 2, "kv must be 6-D");
  TORCH_CHECK(src_pages.is_cuda() && dst_pages.is_cuda() &&
                  src_pages.scalar_type() == torch::kInt32 &&
                  dst_pages.scalar_type() == torch::kInt32,
              "page lists must be int32 on GPU");
  TORCH_CHECK(src_pages.numel() == dst_pages.numel(), "page count mismatch");
  const int n_pages = src_pages.numel();
  if (n_pages == 0) return;
  const int layers = src_kv.size(0);
  const long Ps = src_kv.size(2);
  const long chunk_elems = src_kv.size(3) * src_kv.size(4) * src_kv.size(5);
  TORCH_CHECK(chunk_elems % 8 == 0, "chunk must be 16B-aligned");
  const long chunk_vec = chunk_elems / 8;  // uint4 = 8 bf16
  launch_kv_peer_copy(reinterpret_cast<void*>(dst_base), src_kv.data_ptr(),
                      src_pages.data_ptr(), dst_pages.data_ptr(), n_pages,
                      2 * layers, (int)chunk_vec, chunk_vec,
                      chunk_vec, Ps * chunk_vec, dst_num_pages * chunk_vec,
                      current_stream());
}

// ---- one-shot xGMI all-reduce (parallel/xgmi_allreduce.py) ---------------
// Data buffer: ordinary hipMalloc (IPC-exportable base).  Signal buffer:
// UNCACHED device memory so remote flag stores are immediately visible to
// the local spin loops.

int64_t ar_alloc_signals() {
  void* ptr = nullptr;
  hipError_t err = hipExtMallocWithFlags(
      &ptr, (size_t)xgmi_allreduce_signal_bytes(), hipDeviceMallocUncached);
  TORCH_CHECK(err == hipSuccess,
              "uncached signal alloc failed: ", hipGetErrorString(err));
  (void)hipMemset(ptr, 0, (size_t)xgmi_allreduce_signal_bytes());
  (void)hipDeviceSynchronize();
  return reinterpret_cast<int64_t>(ptr);
}

py::bytes ar_export_ptr(int64_t ptr) {
  hipIpcMemHandle_t handle;
  hipError_t err =
      hipIpcGetMemHandle(&handle, reinterpret_cast<void*>(ptr));
  TORCH_CHECK(err == hipSuccess,
              "hipIpcGetMemHandle failed: ", hipGetErrorString(err));
  return py::bytes(reinterpret_cast<const char*>(&handle), sizeof(handle));
}

unsigned ar_error_flag(int64_t sig_ptr) {
  unsigned err_word = 0;
  // offsetof, NOT sizeof-4: the 128-byte struct alignment pads the tail,
  // so sizeof-4 read the padding and timeouts were invisible (r2 GPU run)
  char* base = reinterpret_cast<char*>(sig_ptr);
  (void)hipMemcpy(&err_word, base + xgmi_allreduce_error_offset(),
                  sizeof(unsigned), hipMemcpyDeviceToHost);
  return err_word;
}

torch::Tensor ar_dump_signals(int64_t sig_ptr) {
  // debug: the whole Signals block as int32 on CPU
  long n = xgmi_allreduce_signal_bytes() / 4;
  auto t = torch::empty({n}, torch::TensorOptions().dtype(torch::kInt32));
  (void)hipMemcpy(t.data_ptr(), reinterpret_cast<void*>(sig_ptr), n * 4,
                  hipMemcpyDeviceToHost);
  return t;
}

torch::Tensor xgmi_allreduce(torch::Tensor inp,
                             std::vector<int64_t> sig_ptrs,
                             std::vector<int64_t> data_ptrs, int64_t rank) {
  check_bf16_contig(inp, "inp");
  const int world = (int)sig_ptrs.size();
  TORCH_CHECK(world >= 1 && world <= 8 &&
                  data_ptrs.size() == (size_t)world && rank >= 0 &&
                  rank < world,
              "bad world/rank");
  TORCH_CHECK(inp.numel() % 8 == 0, "numel must be a multiple of 8");
  auto out = torch::empty_like(inp);
  void* sp[8];
  void* dp[8];
  for (int i = 0; i < world; ++i) {
    sp[i] = reinterpret_cast<void*>(sig_ptrs[i]);
    dp[i] = reinterpret_cast<void*>(data_ptrs[i]);
  }
  launch_xgmi_allreduce(out.data_ptr(), inp.data_ptr(), sp, dp, world,
                        (int)rank, (long)inp.numel(), current_stream());
  return out;
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("rmsnorm", &rmsnorm, "RMSNorm (bf16)");
  m.def("fused_add_rmsnorm", &fused_add_rmsnorm, "x,residual += ; rmsnorm");
  m.def("embed_rows", &embed_rows, "rows of an embedding table");
  m.def("silu_mul", &silu_mul, "silu(gate)*up");
  m.def("rope_store_kv", &rope_store_kv, "RoPE + paged KV write");
  m.def("decode_attention", &decode_attention, "paged flash-decode",
        py::arg("q"), py::arg("key_cache"), py::arg("value_cache"),
        py::arg("block_tables"), py::arg("context_lens"), py::arg("scale"),
        py::arg("num_splits"), py::arg("wide"), py::arg("span") = 128,
        py::arg("tickets") = c10::nullopt);
  m.def("rows_at", &rows_at, "rows that the host names");
  m.def("place_host_inputs", &place_host_inputs, "a decode step's inputs to their place");
  m.def("host_memory", [](torch::Tensor host) {
    return std::make_tuple(fine_grained(host), held_for_stream(host));
  }, "whether kernels read it as it is, and torch keeps it for them");
  m.def("prefill_plan", &prefill_plan, "prompt attention's workgroups",
        py::call_guard<py::gil_scoped_release>());
  m.def("decode_heads", &decode_heads, "rope_heads and decode_attention");
  m.def("prompt_attention_block", &prompt_attention_block,
        "norm, attention and output product of prompts");
  m.def("swiglu_block", &swiglu_block, "norm and gated MLP of many rows");
  m.def("prefill_attention", &prefill_attention, "varlen causal flash prefill");
  m.def("prefill_flash", &prefill_flash, "causal attention of prompts",
        py::arg("q"), py::arg("k"), py::arg("v"), py::arg("block_info"),
        py::arg("seq_lens"), py::arg("scale"),
        py::arg("slots") = c10::nullopt,
        py::arg("items") = c10::nullopt, py::arg("joins") = c10::nullopt,
        py::arg("parts") = 0);
  m.def("mfma_probe", &mfma_probe, "MFMA layout probe");
  m.def("mfma_probe32", &mfma_probe32, "32x32x16 MFMA layout probe");
  m.def("skinny_gemm", &skinny_gemm, "decode-shape GEMM (M<=256)",
        py::arg("a"), py::arg("w"), py::arg("force_splits") = 0,
        py::arg("wide") = false);
  m.def("skinny_parts", &skinny_parts, "decode GEMM as its parts' sums");
  m.def("skinny_swiglu", &skinny_swiglu, "decode gate/up GEMM with silu");
  m.def("tile_swiglu", &tile_swiglu, "gate/up GEMM of a prompt with silu");
  m.def("tile_parts", &tile_parts, "GEMM of a prompt, perhaps as parts' sums");
  m.def("tile_f32", &tile_f32, "GEMM of a prompt with its result in f32");
  m.def("tile_form", &tile_form, "one form of these");
  m.def("tile_split", &tile_split, "the parts of tile_parts");
  m.def("norm_rows", &norm_rows, "norm, GEMM of a few rows and its end");
  m.def("stream_swiglu", &stream_swiglu, "gate/up GEMM of a few rows with silu");
  m.def("stream_linear", &stream_linear, "GEMM of a few rows",
        py::arg("a"), py::arg("w"), py::arg("end") = 0);
  m.def("add_rmsnorm", &add_rmsnorm, "residual += x; its RMS norm");
  m.def("rope_heads", &rope_heads, "head norms, RoPE, paged store");
  // gil_scoped_release on the IPC/copy entry points: mapping or launching
  // against a dying peer can block inside the HIP runtime, and holding the
  // GIL there freezes heartbeats until the controller kills the process
  m.def("ipc_alloc_bf16", &ipc_alloc_bf16,
        "hipMalloc-backed bf16 tensor (IPC-exportable base allocation)",
        py::call_guard<py::gil_scoped_release>());
  m.def("kv_ipc_export", &kv_ipc_export, "hipIpcGetMemHandle of a KV pool");
  m.def("kv_ipc_open", &kv_ipc_open,
        "map a peer KV pool (lazy xGMI peer access)",
        py::call_guard<py::gil_scoped_release>());
  m.def("kv_ipc_close", &kv_ipc_close, "unmap a peer KV pool",
        py::call_guard<py::gil_scoped_release>());
  m.def("kv_peer_copy", &kv_peer_copy,
        "gather local pages -> scatter into peer pool over xGMI",
        py::call_guard<py::gil_scoped_release>());
  m.def("ar_alloc_signals", &ar_alloc_signals,
        "uncached signal buffer for the xGMI all-reduce");
  m.def("ar_export_ptr", &ar_export_ptr, "hipIpc handle of a raw pointer");
  m.def("ar_error_flag", &ar_error_flag, "read the all-reduce error word");
  m.def("ar_dump_signals", &ar_dump_signals, "debug: dump the signal block");
  m.def("ar_counter_offset", &xgmi_allreduce_counter_offset);
  m.def("xgmi_allreduce", &xgmi_allreduce,
        "one-shot all-reduce over peer-mapped HBM (graph-capturable)");
}
