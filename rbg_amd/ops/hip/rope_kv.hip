// Fused RoPE + paged-KV write (gfx950).
//
// One kernel applies rotary embedding (Llama rotate-half / NeoX style) to Q
// and K in place AND scatters the rotated K and V rows into the paged KV
// pool — the write is fused into the producing kernel so K/V never make an
// extra HBM round trip (guide: fuse elementwise work into the producer).
// cos/sin come from a host-precomputed table (guide Appendix B: on-device
// sinf/cosf turns this memory-bound op VALU-bound).
//
// Capability analog: RoPE + KV-cache insert of the engines the reference
// orchestrates.
#include "common.h"

namespace {

// grid.x = tokens; block = 256.  Each block rotates all Q heads + K heads of
// one token and writes K/V to cache[slot].
__global__ void rope_store_kv_kernel(
    __hip_bfloat16* __restrict__ q,          // [T, QH*D]
    __hip_bfloat16* __restrict__ k,          // [T, KVH*D]
    const __hip_bfloat16* __restrict__ v,    // [T, KVH*D]
    __hip_bfloat16* __restrict__ key_cache,  // [pages, KVH, page, D]
    __hip_bfloat16* __restrict__ val_cache,  // [pages, KVH, page, D]
    const float* __restrict__ cos_sin,       // [max_pos, D] = [cos(D/2)|sin(D/2)]
    const int* __restrict__ positions,       // [T]
    const int* __restrict__ slot_mapping,    // [T] page*page_size+off; -1 skip
    const int num_q_heads, const int num_kv_heads, const int head_dim,
    const int page_size,
    const int q_stride, const int kv_stride) { // token-row strides (elems):
  // q/k/v may be SLICES of the fused QKV projection (row pitch = the full
  // qkv width) — strided access here removes three .contiguous() copies
  // per layer (profiles: ~73 ms/bench of pure copy kernels)
  const int token = blockIdx.x;
  const int tid = threadIdx.x;
  const int pos = positions[token];
  const int slot = slot_mapping[token];
  const int half = head_dim / 2;
  const float* cs = cos_sin + (size_t)pos * head_dim;

  // ---- rotate Q: num_q_heads * half pairs -------------------------------
  __hip_bfloat16* q_tok = q + (size_t)token * q_stride;
  const int q_pairs = num_q_heads * half;
  for (int i = tid; i < q_pairs; i += blockDim.x) {
    const int h = i / half, d = i % half;
    __hip_bfloat16* base = q_tok + h * head_dim;
    const float x1 = bf2f(base[d]), x2 = bf2f(base[d + half]);
    const float c = cs[d], s = cs[half + d];
    base[d] = f2bf(x1 * c - x2 * s);
    base[d + half] = f2bf(x2 * c + x1 * s);
  }

  // ---- rotate K and scatter K,V into the paged pool ---------------------
  __hip_bfloat16* k_tok = k + (size_t)token * kv_stride;
  const __hip_bfloat16* v_tok = v + (size_t)token * kv_stride;
  const int page = slot >= 0 ? slot / page_size : 0;
  const int poff = slot >= 0 ? slot % page_size : 0;
  const int kv_pairs = num_kv_heads * half;
  for (int i = tid; i < kv_pairs; i += blockDim.x) {
    const int h = i / half, d = i % half;
    __hip_bfloat16* base = k_tok + h * head_dim;
    const float x1 = bf2f(base[d]), x2 = bf2f(base[d + half]);
    const float c = cs[d], s = cs[half + d];
    const __hip_bfloat16 r1 = f2bf(x1 * c - x2 * s);
    const __hip_bfloat16 r2 = f2bf(x2 * c + x1 * s);
    base[d] = r1;
    base[d + half] = r2;
    if (slot >= 0) {
      __hip_bfloat16* kdst = key_cache +
          (((size_t)page * num_kv_heads + h) * page_size + poff) * head_dim;
      kdst[d] = r1;
      kdst[d + half] = r2;
    }
  }
  if (slot >= 0) {
    // V: straight copy, vectorized 16B per lane
    const int nvec = num_kv_heads * head_dim / 8;
    for (int i = tid; i < nvec; i += blockDim.x) {
      const int h = (i * 8) / head_dim;
      const int d = (i * 8) % head_dim;
      __hip_bfloat16* vdst = val_cache +
          (((size_t)page * num_kv_heads + h) * page_size + poff) * head_dim;
      *reinterpret_cast<uint4*>(vdst + d) =
          *reinterpret_cast<const uint4*>(v_tok + h * head_dim + d);
    }
  }
}

// Heads of 128 from a fused projection [T, q heads | k heads | v heads]: norm
// of every query and key head (NORM), rotation, paged store.  The projection
// is bf16, changed in place, or (PARTS) the f32 sums that the parts of a split
// GEMM left, [parts, T, width], whose result in bf16 goes to `qkv`: neither a
// reduction nor copies and norms of the slices are launches of their own.
// Eight lanes hold a head, each 8 neighbouring dims and the 8 they rotate
// with: 16-byte accesses, and a norm is three shuffles.
// PARTS: those on their way at a time, of few heads eight, of more one, as there are
// threads enough in fewer registers (us, a loop unrolled eight times / eight / one: 32 + 8
// heads, 64 rows of 8 parts 4.8 / 4.2 / -, 1024 of 2 13.7 / 15.0 / 13.2, 2048 of 2 25.0 /
// 26.7 / 24.7; 64 + 8 heads, 1024 of 2 20.5 / 23.7 / 20.0; of 984 sizes 0.94).
template <int PARTS, bool NORM>
__global__ __launch_bounds__(256) void rope_heads_kernel(
    const float* __restrict__ sums, __hip_bfloat16* __restrict__ q,
    const int parts, const int tokens, const int num_q_heads,
    const int num_kv_heads, const int* __restrict__ positions,
    const float* __restrict__ cos_sin,       // [positions, 128] = cos | sin
    const int q_stride, const int kv_stride, __hip_bfloat16* __restrict__ k,
    __hip_bfloat16* __restrict__ v, const __hip_bfloat16* __restrict__ q_norm,
    const __hip_bfloat16* __restrict__ k_norm, const float eps,
    const int* __restrict__ slot_mapping, const int page_size,
    __hip_bfloat16* __restrict__ key_cache,  // [pages, KVH, page, 128]
    __hip_bfloat16* __restrict__ val_cache) {
  constexpr int D = 128;
  const int heads = num_q_heads + 2 * num_kv_heads;
  const int unit = blockIdx.x * 32 + (threadIdx.x >> 3);
  const int lane = threadIdx.x & 7;
  const bool live = unit < tokens * heads;      // shuffles need every lane
  const int token = live ? unit / heads : tokens - 1;
  const int head = live ? unit % heads : heads - 1;
  const bool is_q = head < num_q_heads;
  const bool is_v = head >= num_q_heads + num_kv_heads;
  const int kvh = head - num_q_heads - (is_v ? num_kv_heads : 0);
  __hip_bfloat16* row =
      is_q ? q + (size_t)token * q_stride + head * D
           : (is_v ? v : k) + (size_t)token * kv_stride + kvh * D;
  const int d = lane * 8;
  float x[2][8];
  if constexpr (PARTS > 0) {
    const float* p = sums + ((size_t)token * heads + head) * D + d;
    const size_t step = (size_t)tokens * heads * D;
    f32x4 t[4] = {};
    add_parts<PARTS>(t, parts, [&](int s, int h) {
      return *reinterpret_cast<const f32x4*>(p + s * step + (h >> 1) * 64 +
                                             (h & 1) * 4);
    });
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 8; ++j) x[h][j] = t[h * 2 + (j >> 2)][j & 3];
  } else {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      Bf16x8U u;
      u.u = *reinterpret_cast<const uint4*>(row + h * 64 + d);
#pragma unroll
      for (int j = 0; j < 8; ++j) x[h][j] = bf2f(u.e[j]);
    }
  }
  if (NORM) {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) ss += x[0][j] * x[0][j] + x[1][j] * x[1][j];
#pragma unroll
    for (int off = 4; off >= 1; off >>= 1) ss += __shfl_xor(ss, off, 64);
    if (!is_v) {
      const float inv = rsqrtf(ss / D + eps);
      const __hip_bfloat16* w = is_q ? q_norm : k_norm;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        Bf16x8U u;
        u.u = *reinterpret_cast<const uint4*>(w + h * 64 + d);
#pragma unroll
        for (int j = 0; j < 8; ++j) x[h][j] *= inv * bf2f(u.e[j]);
      }
    }
  }
  Bf16x8U o[2];
  if (!is_v) {
    const float* cs = cos_sin + (size_t)positions[token] * D + d;
    float co[8], si[8];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      *reinterpret_cast<f32x4*>(co + j * 4) =
          *reinterpret_cast<const f32x4*>(cs + j * 4);
      *reinterpret_cast<f32x4*>(si + j * 4) =
          *reinterpret_cast<const f32x4*>(cs + 64 + j * 4);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      o[0].e[j] = f2bf(x[0][j] * co[j] - x[1][j] * si[j]);
      o[1].e[j] = f2bf(x[1][j] * co[j] + x[0][j] * si[j]);
    }
  } else {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 8; ++j) o[h].e[j] = f2bf(x[h][j]);
  }
  if (!live) return;
  if (PARTS || !is_v) {
    *reinterpret_cast<uint4*>(row + d) = o[0].u;
    *reinterpret_cast<uint4*>(row + 64 + d) = o[1].u;
  }
  const int slot = slot_mapping[token];
  if (!is_q && slot >= 0) {
    __hip_bfloat16* dst =
        (is_v ? val_cache : key_cache) +
        (((size_t)(slot / page_size) * num_kv_heads + kvh) * page_size +
         slot % page_size) * D + d;
    *reinterpret_cast<uint4*>(dst) = o[0].u;
    *reinterpret_cast<uint4*>(dst + 64) = o[1].u;
  }
}

}  // namespace

extern "C" {

// parts == 0: q, k, v are bf16 and changed in place; q_norm may be null
void launch_rope_heads(void* q, void* k, void* v, const void* sums, int parts,
                       const void* q_norm, const void* k_norm, float eps,
                       void* key_cache, void* val_cache, const void* cos_sin,
                       const void* positions, const void* slot_mapping,
                       int tokens, int num_q_heads, int num_kv_heads,
                       int page_size, int q_stride, int kv_stride,
                       hipStream_t stream) {
  const int units = tokens * (num_q_heads + 2 * num_kv_heads);
  const dim3 grid((units + 31) / 32), block(256);
#define RH_GO(PARTS, NORM)                                                  \
  rope_heads_kernel<PARTS, NORM><<<grid, block, 0, stream>>>(               \
      (const float*)sums, (__hip_bfloat16*)q, parts, tokens, num_q_heads,   \
      num_kv_heads, (const int*)positions, (const float*)cos_sin, q_stride, \
      kv_stride, (__hip_bfloat16*)k, (__hip_bfloat16*)v,                    \
      (const __hip_bfloat16*)q_norm, (const __hip_bfloat16*)k_norm, eps,    \
      (const int*)slot_mapping, page_size, (__hip_bfloat16*)key_cache,      \
      (__hip_bfloat16*)val_cache)
  const bool many = units > 4096;
  if (parts && many && q_norm) RH_GO(1, true);
  else if (parts && many) RH_GO(1, false);
  else if (parts && q_norm) RH_GO(8, true);
  else if (parts) RH_GO(8, false);
  else if (q_norm) RH_GO(0, true);
  else RH_GO(0, false);
#undef RH_GO
}

void launch_rope_store_kv(void* q, void* k, const void* v, void* key_cache,
                          void* val_cache, const void* cos_sin,
                          const void* positions, const void* slot_mapping,
                          int tokens, int num_q_heads, int num_kv_heads,
                          int head_dim, int page_size, int q_stride,
                          int kv_stride, hipStream_t stream) {
  dim3 grid(tokens), block(256);
  hipLaunchKernelGGL(rope_store_kv_kernel, grid, block, 0, stream,
                     (__hip_bfloat16*)q, (__hip_bfloat16*)k,
                     (const __hip_bfloat16*)v, (__hip_bfloat16*)key_cache,
                     (__hip_bfloat16*)val_cache, (const float*)cos_sin,
                     (const int*)positions, (const int*)slot_mapping,
                     num_q_heads, num_kv_heads, head_dim, page_size,
                     q_stride, kv_stride);
}

}  // extern "C"
