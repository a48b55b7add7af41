// Varlen causal flash attention for prompts, head size 128, keys and values
// as rows or, behind a past, straight from the pages.
//
// Bound: the matrix cores (4 * 128 operations per pair of tokens) and beside
// them the exponentials: 870 to 910 TFLOP/s at 8192 tokens of 32 heads, where
// the 16-row form this replaces reached 346, and 580 to 630 at 2048, where few
// workgroups have most of the work.  A workgroup is 4 waves of 32 query rows each; tiles
// of 64 keys pass LDS in two buffers, one barrier a tile, the next tile's rows
// in flight meanwhile.  (Forming the next tile's scores beside this tile's
// exponentials, for 28 more registers, measured the same.)
//  * The rows of a workgroup are 128 / group tokens with all the query heads
//    of a key head: fewer rows go to waste at the ends of short sequences and
//    on the diagonal than with 128 tokens of one head.
//  * 32x32x16 products: a wave's 32 rows halve the LDS reads per operation of
//    the 16-row form, which LDS bandwidth bound (290 TFLOP/s).
//  * S^T = K Q^T leaves a lane 16 keys of one query, and those weights are the
//    operand of O^T = V^T P^T as they are, with keys 4h..4h+3, 8+4h.. of 16 in
//    place of 8h..8h+7: probabilities never pass LDS, the softmax exchanges one
//    value per 32 keys.  V is read transposed.
//  * Scale and maximum are one fma per score, and sums are rescaled only when
//    some row's maximum grows.  (Letting scores exceed it by 2^8 would be 1 to
//    2% faster, but the largest weight, 1 here, would then be rounded too.)
#include "mfma_util.h"

namespace {

constexpr int DIM = 128, TILE = 64, WAVES = 4, ROWS = WAVES * 32;
constexpr int THREADS = WAVES * 64;
constexpr int KP = DIM + 8;       // row pitch of K in LDS: no bank conflicts
constexpr float LOW = -1e30f;

typedef __attribute__((ext_vector_type(4))) unsigned int pf_u4;

DEV_INLINE pf_u4 pf_load(const __hip_bfloat16* p) {
  return *reinterpret_cast<const pf_u4*>(p);
}

DEV_INLINE bf16x8 pf_frag(pf_u4 u) {
  union { pf_u4 u; bf16x8 v; } c;
  c.u = u;
  return c.v;
}

DEV_INLINE float pf_add2(__bf16 a, __bf16 b, float sum) {
  const bf16x2 ab = {a, b}, ones = {(__bf16)1.f, (__bf16)1.f};
  return __builtin_amdgcn_fdot2_f32_bf16(ab, ones, sum, false);
}

// PAGED: kv rows are named by `slots` ((page << page_shift) + place) and lie in
// [pages, kv heads, 1 << page_shift, DIM].
template <bool PAGED>
__global__ __launch_bounds__(THREADS, 2) void prefill_flash_kernel(
    __hip_bfloat16* __restrict__ out,        // [T, QH, DIM]
    const __hip_bfloat16* __restrict__ q,    // [T, QH, DIM], rows q_stride
    const __hip_bfloat16* __restrict__ k,    // [Tkv, KVH, DIM], rows kv_stride
    const __hip_bfloat16* __restrict__ v,
    const int* __restrict__ slots,           // [Tkv]
    const int* __restrict__ block_info,      // [blocks, 4]: first query row,
    //   block of ROWS / group queries, first kv row, position of the first
    //   query row
    const int* __restrict__ seq_lens,        // [blocks]: kv rows
    const float scale,                       // to the base of 2, > 0
    const bool negate, const int num_q_heads, const int num_kv_heads,
    const int page_shift, const long q_stride, const long kv_stride,
    const int blocks) {
  // Workgroup i runs on XCD i % 8.  A key head stays on one XCD (or on as few
  // as there are heads for), whose L2 then holds that head's rows only.
  const int group = num_q_heads / num_kv_heads;
  int kvh, blk;
  if (num_kv_heads % 8 == 0) {
    const int per = num_kv_heads / 8, i = blockIdx.x / 8;
    kvh = blockIdx.x % 8 * per + i % per;
    blk = i / per;
  } else if (8 % num_kv_heads == 0) {
    const int xcd = blockIdx.x % 8;
    kvh = xcd % num_kv_heads;
    blk = blockIdx.x / 8 * (8 / num_kv_heads) + xcd / num_kv_heads;
  } else {
    kvh = blockIdx.x % num_kv_heads;
    blk = blockIdx.x / num_kv_heads;
  }
  if (blk >= blocks) return;
  const int tokens = ROWS / group;
  const int q_start = block_info[blk * 4];
  const int q_first = block_info[blk * 4 + 1] * tokens;
  const int kv_start = block_info[blk * 4 + 2];
  const int offset = block_info[blk * 4 + 3];
  const int len = seq_lens[blk];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, h = lane >> 5;

  __shared__ __align__(16) __hip_bfloat16 k_lds[2][TILE * KP];
  // [key / 4][dim / 16][key % 4][dim % 16]
  __shared__ __align__(16) __hip_bfloat16 v_lds[2][TILE * DIM];

  const int q_rows = len - offset;            // of this sequence
  const int in = wave * 32 + c;
  const int my_row = q_first + in / group, qh = kvh * group + in % group;
  const int my_pos = offset + my_row;
  bf16x8 qf[8];
  {
    const __hip_bfloat16* qp =
        q + (size_t)(q_start + min(my_row, q_rows - 1)) * q_stride +
        (size_t)qh * DIM + h * 8;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      pf_u4 u = pf_load(qp + s * 16);
      if (negate) u ^= 0x80008000u;
      qf[s] = pf_frag(u);
    }
  }

  const int last = min(offset + q_first + tokens, len) - 1;   // key needed
  // a sequence of fewer keys than queries has queries before its first key,
  // whose result is 0: a block of only those reads no rows
  const int tiles = last < 0 ? 0 : last / TILE + 1;
  const int wave_first = offset + q_first + wave * 32 / group;
  const int wave_end = offset + q_first + (wave * 32 + 31) / group;
  const int wave_tiles = min(tiles, min(wave_end, len - 1) / TILE + 1);

  // thread: 16 bytes of rows tid / 16 + 16 j of a tile
  const int kr = tid >> 4, kc = (tid & 15) * 8;
  pf_u4 ks[4], vs[4];
  int slot[4];
#define PF_SLOTS(t)                                                        \
  if (PAGED) {                                                             \
    _Pragma("unroll") for (int j = 0; j < 4; ++j)                          \
        slot[j] = slots[kv_start +                                         \
                        min((t) * TILE + kr + j * 16, len - 1)];           \
  }
#define PF_ROWS(t)                                                         \
  _Pragma("unroll") for (int j = 0; j < 4; ++j) {                          \
    size_t at;                                                             \
    if (PAGED)                                                             \
      at = (((((size_t)(slot[j] >> page_shift) * num_kv_heads + kvh)       \
              << page_shift) + (slot[j] & ((1 << page_shift) - 1))) * DIM  \
            + kc);                                                         \
    else                                                                   \
      at = (size_t)(kv_start + min((t) * TILE + kr + j * 16, len - 1)) *   \
               kv_stride + (size_t)kvh * DIM + kc;                         \
    ks[j] = pf_load(k + at);                                               \
    vs[j] = pf_load(v + at);                                               \
  }
  const int k_put = kr * KP + kc;
  const int v_put = ((kr >> 2) * 8 + (kc >> 4)) * 64 + (kr & 3) * 16 + (kc & 8);
#define PF_PUT(b)                                                          \
  _Pragma("unroll") for (int j = 0; j < 4; ++j) {                          \
    *reinterpret_cast<pf_u4*>(k_lds[b] + k_put + j * 16 * KP) = ks[j];     \
    *reinterpret_cast<pf_u4*>(v_lds[b] + v_put + j * 16 * DIM) = vs[j];    \
  }

  f32x16 acc[4];
  float m = LOW, l = 0.f;
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[d][i] = 0.f;

  if (tiles > 0) {
    PF_SLOTS(0)
    PF_ROWS(0)
    PF_SLOTS(min(1, tiles - 1))
    PF_PUT(0)
  }
  // A wave stages rows for the others beyond its own last tile, in a loop of
  // its own: a condition around the sums would have them copied every tile.
#define PF_STAGE(t)                                                        \
  __syncthreads();                                                         \
  PF_ROWS(min((t) + 1, tiles - 1))                                         \
  PF_SLOTS(min((t) + 2, tiles - 1))                                        \
  __builtin_amdgcn_sched_barrier(0);
  int t = 0;
  for (; t < wave_tiles; ++t) {
    const int b = t & 1, base = t * TILE;
    PF_STAGE(t)
    {
      f32x16 s[2];
#pragma unroll
      for (int p = 0; p < 2; ++p) {
#pragma unroll
        for (int i = 0; i < 16; ++i) s[p][i] = 0.f;
        const __hip_bfloat16* kp = k_lds[b] + (p * 32 + c) * KP + h * 8;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          s[p] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              pf_frag(pf_load(kp + e * 16)), qf[e], s[p], 0, 0, 0);
      }
      // lane: query c, keys base + 32 p + i % 4 + 8 (i / 4) + 4 h
      if (base + TILE - 1 > wave_first || base + TILE > len) {
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int key = base + p * 32 + i % 4 + 8 * (i / 4) + 4 * h;
            if (key > my_pos || key >= len) s[p][i] = LOW;
          }
      }
      float top = LOW;
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int i = 0; i < 16; ++i) top = fmaxf(top, s[p][i]);
      top = fmaxf(top, __shfl_xor(top, 32, 64)) * scale;
      if (__any(top > m)) {
        const float m_new = fmaxf(m, top);
        const float fade = __builtin_amdgcn_exp2f(m - m_new);
        m = m_new;
        l *= fade;
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[d][i] *= fade;
      }
      bf16x8 pf[4];               // 16 keys each
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          pf[p * 2 + i / 8][i % 8] = (__bf16)__builtin_amdgcn_exp2f(
              __builtin_fmaf(s[p][i], scale, -m));
        }
      // the sum of the weights as they are used, rounded: an error that the
      // largest share with it cancels
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < 8; i += 2)
          l = pf_add2(pf[e][i], pf[e][i + 1], l);
      // 16 keys x 32 dims: lanes of a half read blocks of 4 keys x 16 dims
      const __hip_bfloat16* vp =
          v_lds[b] + h * 512 + ((lane >> 4) & 1) * 64 + (lane & 15) * 4;
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          union { mf_bf4 u[2]; bf16x8 v; } vf;
          vf.u[0] = tr_read4(vp + e * 2048 + d * 128);
          vf.u[1] = tr_read4(vp + e * 2048 + d * 128 + 1024);
          acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf.v, pf[e], acc[d],
                                                           0, 0, 0);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    PF_PUT(1 - b)
  }
  for (; t < tiles; ++t) {
    PF_STAGE(t)
    PF_PUT(1 - (t & 1))
  }
#undef PF_STAGE
#undef PF_SLOTS
#undef PF_ROWS
#undef PF_PUT

  l += __shfl_xor(l, 32, 64);
  if (my_row < q_rows && in < tokens * group) {
    const float inv = l > 0.f ? 1.f / l : 0.f;
    const bool seen = my_pos >= 0;      // else the sums are of masked scores
    __hip_bfloat16* op =
        out + ((size_t)(q_start + my_row) * num_q_heads + qh) * DIM + 4 * h;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        union { __hip_bfloat16 e[4]; uint2 u; } o;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          o.e[j] = f2bf(seen ? acc[d][i * 4 + j] * inv : 0.f);
        *reinterpret_cast<uint2*>(op + d * 32 + i * 8) = o.u;
      }
  }
}

}  // namespace

extern "C" void launch_prefill_flash(
    void* out, const void* q, const void* k, const void* v, const void* slots,
    const void* block_info, const void* seq_lens, float scale, int blocks,
    int num_q_heads, int num_kv_heads, int page_shift, long q_stride,
    long kv_stride, hipStream_t stream) {
  if (blocks == 0) return;
  const int units = num_kv_heads * blocks;
  const int grid = num_kv_heads % 8 && 8 % num_kv_heads == 0
                       ? (units + 7) / 8 * 8 : units;
  // a scale of 0 would make masked scores 0 as well
  const float base2 = fmaxf(fabsf(scale) * 1.44269504088896f, 1e-20f);
#define PF_GO(PAGED)                                                       \
  prefill_flash_kernel<PAGED><<<dim3(grid), dim3(THREADS), 0, stream>>>(   \
      (__hip_bfloat16*)out, (const __hip_bfloat16*)q,                      \
      (const __hip_bfloat16*)k, (const __hip_bfloat16*)v,                  \
      (const int*)slots, (const int*)block_info, (const int*)seq_lens,     \
      base2, scale < 0.f, num_q_heads, num_kv_heads, page_shift, q_stride, \
      kv_stride, blocks)
  if (slots) PF_GO(true);
  else PF_GO(false);
#undef PF_GO
}
