// Varlen causal flash attention for prompts, head size 128, keys and values
// as rows or, behind a past, straight from the pages.
//
// Bound: the issue of vector instructions beside the matrix cores.  Six of them fit
// into the 32 cycles of a product of 32x32x16, each further one takes 5, an exponential
// 9; a wave's tile of 64 keys has 128 besides its 32 products, 32 of them exponentials,
// and 64 more where a maximum grows.  Matrix cores are busy for 57% of the time, vector
// units for 55, LDS for 29; and power: 1.7 to 1.9 GHz at 8192 tokens of 32 heads, 1060
// TFLOP/s.  So nothing is computed in the loop that can be kept: a lane's offsets, which
// change for the last tile only, took 12 instructions a tile, of pages, then in 64 bits,
// 48 (us: 8192 tokens 526 -> 518, 4 of 2048 160 -> 158.6, 1500 after 9000 in pages 254
// -> 248).  Cards differ by a tenth, and figures are of one card each: this kernel and
// the one before queries passed LDS and offsets were kept, in turn on a third, 8192
// tokens 541 -> 530, 4 of 2048 169 -> 164, 1500 after 9000 261 -> 252.
// A workgroup is 4 waves of 32 query rows each; tiles of 64 keys pass LDS in two
// stages, one barrier a tile.
//  * The rows of a workgroup are 128 / group tokens with all the query heads
//    of a key head: fewer rows go to waste at the ends of short sequences and
//    on the diagonal than with 128 tokens of one head.
//  * 32x32x16 products: a wave's 32 rows halve the LDS reads per operation of
//    the 16-row form, which LDS bandwidth bound (290 TFLOP/s).
//  * S^T = K Q^T leaves a lane 16 keys of one query, and those weights are the
//    operand of O^T = V^T P^T as they are, with keys 4h..4h+3, 8+4h.. of 16 in
//    place of 8h..8h+7: probabilities never pass LDS, the softmax exchanges one
//    value per 64 keys.  V is read transposed.
//  * Scale and maximum are one fma per score, and sums are rescaled only when
//    some row's maximum grows.  (Letting scores exceed it by 2^8 would be 1 to
//    2% faster, but the largest weight, 1 here, would then be rounded too.)
//  * Rows go straight to LDS, to places that no read or load meets a conflict
//    at (through registers, with V's writes in conflict: 8192 tokens 600 us, so
//    550), and between the products, pinned there, stand their operands' reads,
//    several ahead, the next tile's loads and three quarters of the exponentials
//    (550 -> 520, where a workgroup has its CU to itself 1.75 -> 1.2 us a tile; half
//    of the exponentials there 1 to 3% more).  A third workgroup on a CU, V in one
//    stage, needs registers that spill (640).
//  * Query rows come, and results go, by way of LDS: 16 lanes have a row's 256 bytes
//    in one piece.  From and to registers as the products have them every lane of an
//    instruction was in another line, of which a CU takes one a cycle: 1.9 us of a
//    workgroup (64 sequences of 64 tokens, 32 heads of 8, 30.3 -> 24.0 us; 23 of 40 to
//    854 104 -> 95; 37 tokens of 16 heads 7.4 -> 6.7; 8192, on the slowest card, 594 ->
//    590).
//  * Blocks are cut by keys where whole ones would leave CUs idle (ops
//    _cut_prefill), whose sums a second launch adds up: 1500 tokens after 9000
//    294 -> 249 us, 512 after 4000 79 -> 55, 40 after 9000 140 -> 27.
#include <type_traits>

#include "mfma_util.h"

namespace {

constexpr int DIM = 128, TILE = 64, WAVES = 4, ROWS = WAVES * 32;
constexpr int THREADS = WAVES * 64;
constexpr int STAGE = TILE * DIM * 2;     // bytes of a tile of K or V
constexpr int LDS = 4 * STAGE;            // two of each
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

// of a lane and the one 32 away
DEV_INLINE float pf_other_half_max(float x) {
  union { float f; unsigned u; } a, b;
  a.f = x;
  const auto both = __builtin_amdgcn_permlane32_swap(a.u, a.u, false, false);
  a.u = both[0];
  b.u = both[1];
  return fmaxf(a.f, b.f);
}

// 16 bytes per lane from base + off, or from a lane's own address, to 16 * lane
// past the wave's LDS address.  Not the compiler's builtin: it would wait for
// the data before any LDS read.
DEV_INLINE void pf_bring(uint32_t off, const void* base, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\t"
               "global_load_lds_dwordx4 %0, %1"
               :: "v"(off), "s"(base), "s"(lds) : "memory", "m0");
}
DEV_INLINE void pf_bring(const void* at, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\t"
               "global_load_lds_dwordx4 %0, off"
               :: "v"(at), "s"(lds) : "memory", "m0");
}

// where kv rows lie: rows kv_stride apart, of which a tile's offsets are 32 bits
// (FROM_ROWS) or not (FROM_FAR_ROWS), or (FROM_PAGES) named by `slots` ((page <<
// page_shift) + place) in [pages, kv heads, 1 << page_shift, DIM] of 4 GB at most, or
// more (FROM_FAR_PAGES)
enum From { FROM_ROWS, FROM_FAR_ROWS, FROM_PAGES, FROM_FAR_PAGES };

template <int FROM>
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
    const int* __restrict__ items,           // [count, 4]: block, its first and
    //   one past its last tile, where its sums go; null: the blocks, whole
    float* __restrict__ part_o,              // [parts, KVH, 4 waves, 16, 64, 4]
    float* __restrict__ part_ml,             // [parts, KVH, ROWS, 2]
    const float scale,                       // to the base of 2, > 0
    const bool negate, const int num_q_heads, const int num_kv_heads,
    const int page_shift, const long q_stride, const long kv_stride,
    const int count) {
  // Workgroup i runs on XCD i % 8.  A key head stays on one XCD (or on as few
  // as there are heads for), whose L2 then holds that head's rows only.
  const int group = num_q_heads / num_kv_heads;
  int kvh, unit;
  if (num_kv_heads % 8 == 0) {
    const int per = num_kv_heads / 8, i = blockIdx.x / 8;
    kvh = blockIdx.x % 8 * per + i % per;
    unit = i / per;
  } else if (8 % num_kv_heads == 0) {
    const int xcd = blockIdx.x % 8;
    kvh = xcd % num_kv_heads;
    unit = blockIdx.x / 8 * (8 / num_kv_heads) + xcd / num_kv_heads;
  } else {
    kvh = blockIdx.x % num_kv_heads;
    unit = blockIdx.x / num_kv_heads;
  }
  if (unit >= count) return;
  const int blk = items ? items[unit * 4] : unit;
  const int part = items ? items[unit * 4 + 3] : -1;
  const int tokens = ROWS / group;
  const int q_start = block_info[blk * 4];
  const int q_first = block_info[blk * 4 + 1] * tokens;
  const int kv_start = block_info[blk * 4 + 2];
  const int offset = block_info[blk * 4 + 3];
  const int len = seq_lens[blk];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, h = lane >> 5;

  // two stages of K, two of V, each [key / 4][16-byte pieces of 4 keys], a piece
  // of V at dim / 16 * 8 + key % 4 * 2 + dim / 8 % 2, of K there with two bits
  // turned over by those of key / 4: no bank conflicts
  extern __shared__ __align__(16) char pf_lds[];

  const int q_rows = len - offset;            // of this sequence
  const float per_group = __builtin_amdgcn_rcpf((float)group);
  // token and head of a row: exact, a quotient is 1 / 256 from a whole number at least
  auto token_of = [&](int row) { return (int)(((float)row + 0.5f) * per_group); };
  const int in = wave * 32 + c;
  const int my_pos = offset + q_first + token_of(in);

  const int last = min(offset + q_first + tokens, len) - 1;   // key needed
  // a sequence of fewer keys than queries has queries before its first key,
  // whose result is 0: a block of only those reads no rows
  const int all = last < 0 ? 0 : last / TILE + 1;
  const int begin = items ? items[unit * 4 + 1] : 0;
  const int tiles = items ? min(all, items[unit * 4 + 2]) : all;
  const int wave_first = offset + q_first + wave * 32 / group;
  const int wave_end = offset + q_first + (wave * 32 + 31) / group;
  const int wave_tiles = min(tiles, min(wave_end, len - 1) / TILE + 1);
  const int whole = min(wave_tiles, max(min(wave_first + 1, len), 0) / TILE);

  // A wave's load brings 4 keys, wave * 4 + 16 j .. of a tile; a lane's piece
  // of its key's 16
  const int kr = wave * 4 + ((lane >> 1) & 3);
  const uint32_t v_piece = ((lane >> 3) * 2 + (lane & 1)) * 16;
  const uint32_t k_piece = (((lane >> 3) ^ (wave & 1)) * 2 +
                            ((lane & 1) ^ (wave >> 1))) * 16;
  const uint32_t lds0 = (uint32_t)(uintptr_t)pf_lds + wave * 1024;
  const size_t row_bytes = (size_t)kv_stride * 2;
  constexpr bool PAGED = FROM == FROM_PAGES || FROM == FROM_FAR_PAGES;
  const uint32_t head_rows = (uint32_t)kvh << page_shift;
  const size_t head_at = PAGED ? (size_t)head_rows * DIM
                               : (size_t)kvh * DIM + (size_t)kv_start * kv_stride;
  const char* const kb = (const char*)(k + head_at);
  const char* const vb = (const char*)(v + head_at);
  // rows of a page beyond those of one head
  const uint32_t beside = (uint32_t)(num_kv_heads - 1) << page_shift;
  // A lane's offsets in a tile change only for the last, whose rows past the
  // sequence's are its last one: addresses would be a tenth of the VALU's work.
  const int ragged = all * TILE > len ? all - 1 : -1;
  uint32_t k_off[4], v_off[4];      // of a tile's rows
  uint32_t s_off[4];                // of its slots
  auto aim = [&](int t) {
    if (FROM == FROM_ROWS)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = t == ragged ? min(kr + j * 16, len - 1 - t * TILE)
                                  : kr + j * 16;
        k_off[j] = __umul24(r, (uint32_t)row_bytes) + k_piece;
        v_off[j] = __umul24(r, (uint32_t)row_bytes) + v_piece;
      }
  };
  auto aim_slots = [&](int t) {
    if (PAGED)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        s_off[j] = (t == ragged ? min(kr + j * 16, len - 1 - t * TILE)
                                : kr + j * 16) * 4;
  };
  uint32_t slot[4] = {};                    // of the next tile
  auto name = [&](int t, bool plain = false) {
    if (!PAGED) return;
    if (!plain && t == ragged) aim_slots(t);
    const char* at = (const char*)(slots + kv_start + t * TILE);
#pragma unroll
    for (int j = 0; j < 4; ++j) slot[j] = *(const uint32_t*)(at + s_off[j]);
  };
  // the compiler's wait for them, which counts only its own loads, comes here; then
  // the rows that they name
  auto named = [&]() {
    if (!PAGED) return;
#pragma unroll
    for (int j = 0; j < 4; ++j) asm volatile("" : "+v"(slot[j]));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t page = slot[j] >> page_shift;
      if (FROM == FROM_FAR_PAGES) {
        k_off[j] = page;
        v_off[j] = slot[j];
      } else {
        uint32_t row;       // both factors are of 24 bits, as rows are
        asm("v_mad_u32_u24 %0, %1, %2, %3"
            : "=v"(row) : "v"(page), "s"(beside), "v"(slot[j]));
        k_off[j] = row * (DIM * 2) + k_piece;
        v_off[j] = row * (DIM * 2) + v_piece;
      }
    }
  };
  auto bring = [&](int j, const char* base, int t, bool of_v, uint32_t to) {
    if (FROM == FROM_FAR_PAGES) {
      pf_bring(base + (of_v ? v_piece : k_piece) +
                   ((size_t)k_off[j] * beside + v_off[j]) * (DIM * 2),
               to + j * 4096);
    } else if (FROM == FROM_PAGES) {
      pf_bring(of_v ? v_off[j] : k_off[j], base, to + j * 4096);
    } else if (FROM == FROM_ROWS) {
      pf_bring(of_v ? v_off[j] : k_off[j], base + t * TILE * row_bytes,
               to + j * 4096);
    } else {
      const int r = min(kr + j * 16, len - 1 - t * TILE);
      pf_bring(base + (t * TILE + r) * row_bytes + (of_v ? v_piece : k_piece),
               to + j * 4096);
    }
  };
  // all of tile `t`, or the q-th of its 8 loads, to the stages of tile `as`
  auto bring_one = [&](int q, int t, int as) {
    const uint32_t to = lds0 + (as & 1) * STAGE;
    if (q & 1) bring(q >> 1, vb, t, true, to + 2 * STAGE);
    else bring(q >> 1, kb, t, false, to);
  };
  auto bring_all = [&](int t, int as) {
#pragma unroll
    for (int q = 0; q < 8; ++q) bring_one(q, t, as);
  };

  // A wave's own 8 KB of a stage, which no other wave's loads go to: row r of 32 at
  // its place, piece p of 16 at p ^ r % 16
  auto own = [&](int j, int as) {             // rows 4 j ..
    return wave * 1024 + (as & 1) * STAGE + (j & 3) * 4096 + (j >> 2) * 2 * STAGE;
  };

  // this lane's key and piece of K: row p * 32 + c, dims e * 16 + h * 8 ..
  const int kblk = c >> 2;
  const int k_at = kblk * 1024 + (c & 3) * 32 + ((h ^ ((kblk >> 1) & 1)) * 16);
  const int k_even = k_at + (kblk & 1) * 128, k_odd = k_at - (kblk & 1) * 128;
  const int v_at = 2 * STAGE + h * 1024 + ((lane >> 4) & 1) * 128 +
                   (lane & 15) * 8;

  f32x16 acc[4];
  float m = LOW, l = 0.f;
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[d][i] = 0.f;

  bf16x8 qf[8];
  if (begin < tiles) {
    aim(begin);
    aim_slots(begin);
    name(begin);
    named();
    // the rows of q in whole lines, by way of the stage that comes second
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int r = wave * 32 + j * 4 + (lane >> 4), token = token_of(r);
      pf_bring(q + (size_t)(q_start + min(q_first + token, q_rows - 1)) * q_stride +
                   (size_t)(kvh * group + r - token * group) * DIM +
                   ((lane & 15) ^ (r & 15)) * 8,
               (uint32_t)(uintptr_t)pf_lds + own(j, begin + 1));
    }
    bring_all(begin, begin);
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      pf_u4 u = *reinterpret_cast<const pf_u4*>(
          pf_lds + own(0, begin + 1) + ((c >> 2) & 3) * 4096 +
          (c >> 4) * 2 * STAGE + (c & 3) * 256 + (((s * 2 + h) ^ (c & 15)) * 16));
      if (negate) u ^= 0x80008000u;
      qf[s] = pf_frag(u);
    }
    name(min(begin + 1, tiles - 1));
  }
  // Waited for here: the compiler would wait for them in every tile.
#pragma unroll
  for (int s = 0; s < 8; ++s) asm volatile("" : "+v"(qf[s]));
  const int seen_to = min(my_pos, len - 1) - 4 * h;   // the last key, of a lane's
#define PF_MEET()                                                          \
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); \
  named();
  // One tile's products.  Between them, one thing at a time and pinned there,
  // stand the reads of their operands ahead of them, the next tile's loads and
  // three quarters of the exponentials.
  auto products = [&](auto masked, int t) {
    constexpr bool MASK = decltype(masked)::value;
    const int base = t * TILE, next = min(t + 1, tiles - 1);
    if (MASK && next == ragged) aim(next);
    const char* kp = pf_lds + (t & 1) * STAGE;
    const __hip_bfloat16* vp =
        (const __hip_bfloat16*)(pf_lds + v_at + (t & 1) * STAGE);
    auto k_read = [&](int n) {
      return pf_frag(*reinterpret_cast<const pf_u4*>(
          kp + (n & 1 ? k_odd : k_even) + (n >> 3) * 8192 + (n & 7) * 128));
    };
    // 16 keys x 32 dims: lanes of a half read blocks of 4 keys x 16 dims
    auto v_read = [&](int n) {
      union { mf_bf4 u[2]; bf16x8 v; } f;
      const __hip_bfloat16* at = vp + (n >> 2) * 2048 + (n & 3) * 128;
      f.u[0] = tr_read4(at);
      f.u[1] = tr_read4(at + 1024);
      return f.v;
    };
    constexpr int AHEAD = 6, V_AHEAD = 4;
    bf16x8 kf[AHEAD], vf[V_AHEAD];
    f32x16 s[2] = {};
    float top = LOW;
#pragma unroll
    for (int n = 0; n < AHEAD; ++n) kf[n] = k_read(n);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < 16; ++n) {
      s[n >> 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          kf[n % AHEAD], qf[n & 7], s[n >> 3], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (n + AHEAD < 16) kf[n % AHEAD] = k_read(n + AHEAD);
      else if (n + V_AHEAD >= 16) vf[n + V_AHEAD - 16] = v_read(n + V_AHEAD - 16);
      if (n < 8) bring_one(n, next, t + 1);
      if (!MASK && n >= 10 && n < 15) {
#pragma unroll
        for (int i = (n - 10) * 3; i < min(16, (n - 9) * 3 + (n == 14)); ++i)
          top = fmaxf(top, s[0][i]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    name(min(t + 2, tiles - 1), !MASK);
    // lane: query c, keys base + 32 p + i % 4 + 8 (i / 4) + 4 h
    if (MASK) {
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          if (p * 32 + i % 4 + 8 * (i / 4) > seen_to - base) s[p][i] = LOW;
          if (p == 0) top = fmaxf(top, s[0][i]);
        }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) top = fmaxf(top, s[1][i]);
    top = pf_other_half_max(top) * scale;
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
    auto weigh = [&](int n) {
      pf[n >> 3][n & 7] = (__bf16)__builtin_amdgcn_exp2f(
          __builtin_fmaf(s[n >> 4][n & 15], scale, -m));
    };
#pragma unroll
    for (int n = 0; n < 8; ++n) weigh(n);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < 16; ++n) {
      acc[n & 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          vf[n % V_AHEAD], pf[n >> 2], acc[n & 3], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (n + V_AHEAD < 16) vf[n % V_AHEAD] = v_read(n + V_AHEAD);
      if (n < 12) {
        weigh(8 + 2 * n);
        weigh(9 + 2 * n);
      } else {
        // the sum of the weights as they are used, rounded: an error that the
        // largest share with it cancels
#pragma unroll
        for (int i = 0; i < 8; i += 2)
          l = pf_add2(pf[n - 12][i], pf[n - 12][i + 1], l);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int t = begin;
  // what it loads and names ahead is not the ragged tile
  const int plain = ragged < 0 ? whole : min(whole, ragged - (PAGED ? 2 : 1));
  for (; t < plain; ++t) {
    PF_MEET()
    products(std::false_type(), t);
  }
  for (; t < wave_tiles; ++t) {
    PF_MEET()
    products(std::true_type(), t);
  }
  // beyond its own last tile a wave brings rows for the others
  for (; t < tiles; ++t) {
    PF_MEET()
    if (min(t + 1, tiles - 1) == ragged) aim(ragged);
    bring_all(min(t + 1, tiles - 1), t + 1);
    name(min(t + 2, tiles - 1));
  }
#undef PF_MEET
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // LDS is in use until then

  l += __shfl_xor(l, 32, 64);
  if (part >= 0) {
    const size_t at = ((size_t)part * num_kv_heads + kvh) * ROWS;
#pragma unroll
    for (int e = 0; e < 16; ++e)
      *reinterpret_cast<f32x4*>(
          part_o + at * DIM + ((wave * 16 + e) * 64 + lane) * 4) =
          f32x4{acc[e >> 2][(e & 3) * 4], acc[e >> 2][(e & 3) * 4 + 1],
                acc[e >> 2][(e & 3) * 4 + 2], acc[e >> 2][(e & 3) * 4 + 3]};
    if (h == 0) {
      part_ml[(at + in) * 2] = m;
      part_ml[(at + in) * 2 + 1] = l;
    }
    return;
  }
  // Rows as whole lines, by way of the wave's own part of the stage that no tile is in:
  // the last barrier has passed since others read it, and its own loads to it are
  // there.  A lane and the one 32 away make up 16 bytes of two pieces.
  const float inv = l > 0.f ? 1.f / l : 0.f;
  const bool seen = my_pos >= 0;        // else the sums are of masked scores
  char* const mine = pf_lds + own(0, tiles);
#pragma unroll
  for (int n = 0; n < 8; ++n) {         // dims 16 n ..
    union { __hip_bfloat16 e[4]; unsigned u[2]; } a, b;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      a.e[j] = f2bf(seen ? acc[n >> 1][(n & 1) * 8 + j] * inv : 0.f);
      b.e[j] = f2bf(seen ? acc[n >> 1][(n & 1) * 8 + 4 + j] * inv : 0.f);
    }
    const auto x = __builtin_amdgcn_permlane32_swap(a.u[0], b.u[0], false, false);
    const auto y = __builtin_amdgcn_permlane32_swap(a.u[1], b.u[1], false, false);
    *reinterpret_cast<pf_u4*>(mine + ((c >> 2) & 3) * 4096 + (c >> 4) * 2 * STAGE +
                              (c & 3) * 256 + (((n * 2 + h) ^ (c & 15)) * 16)) =
        pf_u4{x[0], y[0], x[1], y[1]};
  }
  // lanes read what others of the wave wrote: in that order for the compiler too
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int row = j * 4 + (lane >> 4), r = wave * 32 + row, token = token_of(r);
    const pf_u4 u = *reinterpret_cast<const pf_u4*>(
        pf_lds + own(j, tiles) + (lane >> 4) * 256 +
        (((lane & 15) ^ (row & 15)) * 16));
    if (q_first + token < q_rows && r < tokens * group)
      *reinterpret_cast<pf_u4*>(
          out + ((size_t)(q_start + q_first + token) * num_q_heads + kvh * group +
                 r - token * group) * DIM + (lane & 15) * 8) = u;
  }
}

// The sums of a block whose keys were cut, from those of its parts.  A workgroup
// per block, key head and 32 dims; bound by reading them, 512 bytes a row and
// part, in the order in which the kernel above holds them.
__global__ __launch_bounds__(THREADS) void prefill_join_kernel(
    __hip_bfloat16* __restrict__ out, const float* __restrict__ part_o,
    const float* __restrict__ part_ml, const int* __restrict__ block_info,
    const int* __restrict__ seq_lens,
    const int* __restrict__ joins,           // [n, 3]: block, its first part, parts
    const int num_q_heads, const int num_kv_heads) {
  const int blk = joins[blockIdx.x * 3], first = joins[blockIdx.x * 3 + 1];
  const int parts = joins[blockIdx.x * 3 + 2];
  const int kvh = blockIdx.y, d = blockIdx.z;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 31, h = lane >> 5, in = wave * 32 + c;
  const int group = num_q_heads / num_kv_heads, tokens = ROWS / group;
  const int offset = block_info[blk * 4 + 3];
  const int my_row = block_info[blk * 4 + 1] * tokens + in / group;
  float top = LOW, l = 0.f;
  f32x4 o[4] = {};
  for (int p = 0; p < parts; ++p) {
    const size_t at = ((size_t)(first + p) * num_kv_heads + kvh) * ROWS;
    f32x4 x[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      x[e] = *reinterpret_cast<const f32x4*>(
          part_o + at * DIM + ((wave * 16 + d * 4 + e) * 64 + lane) * 4);
    const float m = part_ml[(at + in) * 2];
    const float most = fmaxf(top, m);
    const float fade = __builtin_amdgcn_exp2f(top - most);
    const float f = __builtin_amdgcn_exp2f(m - most);
    top = most;
    l = l * fade + part_ml[(at + in) * 2 + 1] * f;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = o[e] * fade + x[e] * f;
  }
  if (my_row >= seq_lens[blk] - offset || in >= tokens * group) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  const bool seen = offset + my_row >= 0;
  __hip_bfloat16* op = out +
      ((size_t)(block_info[blk * 4] + my_row) * num_q_heads + kvh * group +
       in % group) * DIM + d * 32 + 4 * h;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    union { __hip_bfloat16 e[4]; uint2 u; } b;
#pragma unroll
    for (int j = 0; j < 4; ++j) b.e[j] = f2bf(seen ? o[e][j] * inv : 0.f);
    *reinterpret_cast<uint2*>(op + e * 8) = b.u;
  }
}

}  // namespace

// items and joins: null, or the blocks' work as cut up and what is to be joined;
// kv_rows: of all pages and heads, where there are slots
extern "C" void launch_prefill_flash(
    void* out, const void* q, const void* k, const void* v, const void* slots,
    const void* block_info, const void* seq_lens, float scale, int blocks,
    const void* items, int count, const void* joins, int joined, void* part_o,
    void* part_ml, int num_q_heads, int num_kv_heads, int page_shift,
    long q_stride, long kv_stride, long kv_rows, hipStream_t stream) {
  if (!items) count = blocks;
  if (count == 0) return;
  const int units = num_kv_heads * count;
  const int grid = num_kv_heads % 8 && 8 % num_kv_heads == 0
                       ? (units + 7) / 8 * 8 : units;
  // a scale of 0 would make masked scores 0 as well
  const float base2 = fmaxf(fabsf(scale) * 1.44269504088896f, 1e-20f);
#define PF_GO(FROM)                                                        \
  prefill_flash_kernel<FROM><<<dim3(grid), dim3(THREADS), LDS, stream>>>(  \
      (__hip_bfloat16*)out, (const __hip_bfloat16*)q,                      \
      (const __hip_bfloat16*)k, (const __hip_bfloat16*)v,                  \
      (const int*)slots, (const int*)block_info, (const int*)seq_lens,     \
      (const int*)items, (float*)part_o, (float*)part_ml, base2,           \
      scale < 0.f, num_q_heads, num_kv_heads, page_shift, q_stride,        \
      kv_stride, count)
  if (slots && kv_rows <= 1 << 24) PF_GO(FROM_PAGES);
  else if (slots) PF_GO(FROM_FAR_PAGES);
  else if (kv_stride < (1 << 23)) PF_GO(FROM_ROWS);
  else PF_GO(FROM_FAR_ROWS);
#undef PF_GO
  if (joined)
    prefill_join_kernel<<<dim3(joined, num_kv_heads, DIM / 32), dim3(THREADS),
                          0, stream>>>(
        (__hip_bfloat16*)out, (const float*)part_o, (const float*)part_ml,
        (const int*)block_info, (const int*)seq_lens, (const int*)joins,
        num_q_heads, num_kv_heads);
}
