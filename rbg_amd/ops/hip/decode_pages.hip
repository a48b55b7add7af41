// Paged flash-decode over pages of 16 keys and head size 128: one query token
// per sequence, all query heads of a key head in one pass.
//
// Bound: the keys and values, read once (a plain read reaches 6.1-6.3 TB/s).
//  * A page of one key head is 4 KB in one piece.  Keys go from memory
//    straight into MFMA registers as rows of S^T = K q^T, whose result holds
//    8 keys of one head per lane: softmax needs two shuffles per 32 keys, and
//    its weights are the operand of O^T = V^T P^T as they are, with keys
//    4g..4g+3 of two pages in place of 8g..8g+7.  Only V passes LDS, private
//    to its wave, to be read transposed: no barrier inside the walk.
//  * The next 32 keys and values are in flight while these are used: 16 KB
//    per wave.
//  * Values, read in whole lines and once, are loaded non-temporally (219 ->
//    198 us at 128 x 2080); keys, whose lines two loads share, are not.
//  * Work is cut by keys, not by sequences: every workgroup takes `span` keys
//    of one sequence, whatever the sequence's length, so a batch of ragged
//    lengths fills the chip as a regular one does; longer ones only where the
//    grid has too few for the sequence.  The grid is fixed when a step is
//    captured; workgroups past the end of their sequence leave at once.
//    Few sequences share one workgroup a CU, or two (even_keys): every wave reads all
//    lengths, takes the shortest parts that leave none over, and finds its own among
//    those that have keys.  A CU with two workgroups takes twice as long as the others,
//    and with fixed parts, and workgroups without keys between them, some had two: 7 of
//    300 to 3000 tokens 19.4 -> 14.9 us, 3 of 10500 to 15000 43 -> 33, 20 of 400 to
//    6000 in 24 rows 60 -> 59, 16 of 4000 to 16000 138 -> 123, 31 of 500 and one of
//    16000 81 -> 42, 30 of 400 to 4000 with 2 key heads 26 -> 18.  Over 70 batches it
//    takes 0.85 of the time of fixed parts; eight take longer: six 0.2 to 0.9 us, for
//    the search (7 of 100 6.0 -> 6.2), 11 of 300 to 6000 with 16 key heads 60.0 ->
//    63.4, 25 of up to 4800 with two query heads a key head 60.2 -> 63.2.
//  * With a ticket per (sequence, key head), which the caller keeps and which is
//    0 between launches, the last workgroup of a sequence adds up what its parts
//    left: no launch of its own, which costs 1 to 3 us (1 sequence of 100 keys
//    6.3 -> 4.8 us, 64 of up to 2048 68 -> 65).  Ordered without fences: sums are
//    stored and loaded as atomics at agent scope, which pass the XCD's L2 either
//    way; a wave's stores are there when its vmcnt has counted them off, every
//    wave's before the barrier, and the ticket is drawn behind it; the loads
//    stand behind the barrier after the ticket.  (Release and acquire fences write
//    back and invalidate whole caches: six layers of 3 sequences of up to 15000
//    tokens 871 -> 1715 us, 45 of up to 2500 1125 -> 1934.)
#include "decode_heads.h"
#include "decode_join.h"

namespace {

constexpr int PAGE = 16, WAVES = 4, STEP = 32;
constexpr int VROW = 528;         // of a 16-dim column of 32 values: 512 + pad,
                                  // so that writes of a row meet no conflicts
static_assert(WAVES * STEP == PART_ROUND, "parts are whole rounds");

typedef __attribute__((ext_vector_type(4))) unsigned int dp_u4;

DEV_INLINE dp_u4 dp_load(const __hip_bfloat16* p) {
  return *reinterpret_cast<const dp_u4*>(p);
}

DEV_INLINE bf16x8 dp_frag(dp_u4 u) {
  union { dp_u4 u; bf16x8 v; } c;
  c.u = u;
  return c.v;
}

DEV_INLINE void dp_share(float* to, float x) {
  __hip_atomic_store(to, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

DEV_INLINE f32x2 dp_shared(const float* from) {
  union { unsigned long long u; f32x2 v; } x;
  x.u = __hip_atomic_load((const unsigned long long*)from, __ATOMIC_RELAXED,
                          __HIP_MEMORY_SCOPE_AGENT);
  return x.v;
}

// TOGETHER: all key heads of a (sequence, part) run on one XCD, workgroup i on
// XCD i % 8, which then translates an eighth of the pool's addresses (128
// sequences of 2080 tokens, 8 heads: 198 -> 179 us, 6.1 TB/s).  A small batch
// of ragged lengths would leave XCDs idle (45 of up to 2500: 63 -> 68 us).
// PROJ: the heads come as the projection left them.  Every workgroup adds up,
// norms and rotates its own queries, on the way to LDS, while its keys are on
// theirs; the one with a sequence's last key does the new key and value too, stores
// them, and puts them in place of what registers already hold of that row.  The
// rotation's own launch was 3 us of a layer (six layers, us: 7 sequences of qwen 8b
// 715 -> 700, 45 of 8b 1109 -> 1097, 64 of qwen 32b, four layers, 1282 -> 1275, 128 of
// 8b 2017 -> 2014).  With the parts by the lengths 80 batches of 1 to 256 sequences,
// from bf16 and 1, 5 and 12 parts, take 0.77 of the time of rotation and fixed parts, 25
// of up to 4800 and 11 of 300 to 6000 of the above 1 to 3% more or less, and 256 of 40
// tokens 1.0 to 1.07, as each has a workgroup's start.
template <int QPG, bool TOGETHER, bool PROJ>
__global__ __launch_bounds__(64 * WAVES, 3) void decode_pages_kernel(
    const int* __restrict__ lens,           // [seqs]
    const int kv_heads, const int seqs, const int splits,
    const int most,                         // workgroups of a slot, below
    const int* __restrict__ tables,         // [seqs, max_pages]
    const int max_pages, const int least, const int whole,
    const int slots,                        // a key head's workgroups, or 0
    const __hip_bfloat16* __restrict__ q,   // [seqs, QH, DIM], rows q_stride
    const int q_stride, const float scale,  // to the base of 2
    __hip_bfloat16* keys,                   // [pages, KVH, PAGE, DIM]
    __hip_bfloat16* values,
    float* __restrict__ part_o,             // [splits, seqs, QH, DIM]
    float* __restrict__ part_ml,            // [splits, seqs, QH, 2]
    __hip_bfloat16* __restrict__ out,       // [seqs, QH, DIM]
    int* __restrict__ tickets,              // [seqs, KVH], or null
    const DecodeHeads proj) {
  int kvh = blockIdx.x, seq = blockIdx.y, split = blockIdx.z;
  if (TOGETHER) {
    const int lin = kvh + kv_heads * (seq + seqs * split);
    const int pairs = seqs * splits, group = lin / (8 * kv_heads);
    const int in = lin % (8 * kv_heads);
    const bool whole = (group + 1) * 8 <= pairs;
    const int pair = group * 8 + (whole ? in % 8 : in / kv_heads);
    kvh = whole ? in / 8 : in % kv_heads;
    seq = pair % seqs;
    split = pair / seqs;
  }
  int ctx, span;
  constexpr int JOINS = 64 * WAVES / (QPG * DIM / 4) * 8;    // parts of a round
  if (!TOGETHER && slots && seqs == 1) {
    ctx = lens[0];
    span = even_keys(ctx, slots, JOINS, splits);
    split = blockIdx.y;
    seq = 0;
  } else if (!TOGETHER && slots) {
    const int in = threadIdx.x & 63;
    const int n = in < seqs ? lens[in] : 0;
    int parts, upto;
    span = even_keys(n, seqs, slots, most, JOINS, splits, &parts, &upto);
    const uint64_t later = __ballot(upto > (int)blockIdx.y);
    if (!later) return;
    seq = __builtin_ctzll(later);
    ctx = __builtin_amdgcn_readlane(n, seq);
    split = blockIdx.y - __builtin_amdgcn_readlane(upto - parts, seq);
  } else {
    ctx = lens[seq];
    span = part_keys(ctx, least, whole, splits);
  }
  const int begin = split * span, end = min(ctx, begin + span);
  if (begin >= ctx && split > 0) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int heads = kv_heads * QPG;

  __shared__ __align__(16) __hip_bfloat16 v_lds[WAVES][8 * VROW];
  __shared__ float sums[WAVES][QPG][2];
  __shared__ __align__(16) __hip_bfloat16 heads_lds[PROJ ? QPG + 2 : 1][DIM];
  static_assert(sizeof(v_lds) >= WAVES * QPG * DIM * 4 &&
                    sizeof(v_lds) >= 64 * WAVES * 6 * 4, "merges fit");

  // the heads' queries as columns (QPG of 16), 4 pieces of 32 dims
  bf16x8 qf[4];
  if (!PROJ) {
    const __hip_bfloat16* qp = q + (size_t)seq * q_stride +
                               (size_t)(kvh * QPG + min(c, QPG - 1)) * DIM;
#pragma unroll
    for (int d = 0; d < 4; ++d) qf[d] = dp_frag(dp_load(qp + d * 32 + g * 8));
  }
  const int* table = tables + (size_t)seq * max_pages;
  const int last_page = max(end - 1, 0) / PAGE;
  const size_t head_at = (size_t)kvh * PAGE * DIM;
  const size_t page_size = (size_t)kv_heads * PAGE * DIM;
  const int k_at = c * DIM + g * 8;       // this lane's part of a page of keys
  const int v_at = lane * 8;              // and of values, in 4 pieces of 1 KB
  __hip_bfloat16* vl = v_lds[wave];
  // piece j of a page: key 4j + g, dims 8c..; [dim / 16][page][key][dim % 16]
  const int v_put = (c >> 1) * VROW + g * 16 + (c & 1) * 8;

  f32x4 acc[8];
  float m = LOW, l = 0.f;
#pragma unroll
  for (int t = 0; t < 8; ++t) acc[t] = {0.f, 0.f, 0.f, 0.f};

  dp_u4 kr[2][4], vr[2][4];
#define DP_PAGE(at, p) table[min((at) / PAGE + (p), last_page)]
#define DP_KEYS(page)                                                      \
  _Pragma("unroll") for (int p = 0; p < 2; ++p) {                          \
    const __hip_bfloat16* src = keys + head_at + k_at +                    \
                                (size_t)page[p] * page_size;               \
    _Pragma("unroll") for (int d = 0; d < 4; ++d)                          \
        kr[p][d] = dp_load(src + d * 32);                                  \
  }
#define DP_VALUES(page)                                                    \
  _Pragma("unroll") for (int p = 0; p < 2; ++p) {                          \
    const __hip_bfloat16* src = values + head_at + v_at +                  \
                                (size_t)page[p] * page_size;               \
    _Pragma("unroll") for (int j = 0; j < 4; ++j)                          \
        vr[p][j] = __builtin_nontemporal_load(                             \
            reinterpret_cast<const dp_u4*>(src + j * 512));                \
  }
  int at = begin + wave * STEP;
  int page[2];                    // of the next step, known one step ahead
  int fresh = -1;                 // PROJ: the new key, where this workgroup has it
  if (!PROJ) {
    if (at < end) {
      page[0] = DP_PAGE(at, 0);
      page[1] = DP_PAGE(at, 1);
      DP_KEYS(page)
      DP_VALUES(page)
      page[0] = DP_PAGE(at + WAVES * STEP, 0);
      page[1] = DP_PAGE(at + WAVES * STEP, 1);
    }
  } else {
    // a wave has a head at a time, a lane two dims that rotate into one another;
    // the last key's workgroup has the new ones too, of no keys the first
    constexpr int MINE = (QPG + 2 + WAVES - 1) / WAVES, ROUND = 8;
    const bool keeps = end == ctx || ctx <= 0;
    const int units = keeps ? QPG + 2 : QPG;
    const int parts = proj.parts, slot = proj.slots[seq];
    if (ctx > 0) {
      page[0] = DP_PAGE(at, 0);
      page[1] = DP_PAGE(at, 1);
      if (keeps && slot == table[(ctx - 1) / PAGE] * PAGE + (ctx - 1) % PAGE)
        fresh = ctx - 1;
    } else {
      page[0] = page[1] = 0;
    }
    const float* cs = proj.cos_sin + (size_t)proj.positions[seq] * DIM;
    const float co = cs[lane], si = cs[lane + 64];
    const size_t step = (size_t)seqs * q_stride;
    uint32_t raw[MINE][ROUND][2];
    size_t from[MINE];
#define DP_PART(n, i, s)    /* past the last part: that one, to no use */    \
  do {                                                                     \
    const float* part =                                                    \
        proj.sums + (min(s, parts - 1) * step + from[n]);          \
    raw[n][i][0] = __float_as_uint(part[lane]);                            \
    raw[n][i][1] = __float_as_uint(part[lane + 64]);                       \
  } while (0)
#pragma unroll
    for (int n = 0; n < MINE; ++n) {
      const int u = min(wave + n * WAVES, units - 1);
      const int head = u < QPG ? kvh * QPG + u
                               : heads + (u - QPG) * kv_heads + kvh;
      from[n] = (size_t)seq * q_stride + head * DIM;
      if (parts) {
#pragma unroll
        for (int i = 0; i < ROUND; ++i) DP_PART(n, i, i);
      } else {
        const unsigned short* p = (const unsigned short*)q + from[n];
        raw[n][0][0] = p[lane];
        raw[n][0][1] = p[lane + 64];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // without a condition, which the sums' wait would have to take for none
    DP_KEYS(page)
    DP_VALUES(page)
    __builtin_amdgcn_sched_barrier(0);
    if (ctx > 0) {
      page[0] = DP_PAGE(at + WAVES * STEP, 0);
      page[1] = DP_PAGE(at + WAVES * STEP, 1);
    }
#pragma unroll
    for (int n = 0; n < MINE; ++n) {
      const int u = wave + n * WAVES;
      if (u >= units) break;
      float x[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        x[h] = 0.f;
        if (parts == 0) x[h] = __uint_as_float(raw[n][0][h] << 16);
#pragma unroll
        for (int i = 0; i < ROUND; ++i)
          if (i < parts) x[h] += __uint_as_float(raw[n][i][h]);
      }
      for (int s = ROUND; s < parts; s += 2) {
        DP_PART(n, 0, s);
        DP_PART(n, 1, s + 1);
        x[0] += __uint_as_float(raw[n][0][0]);
        x[1] += __uint_as_float(raw[n][0][1]);
        if (s + 1 < parts) {
          x[0] += __uint_as_float(raw[n][1][0]);
          x[1] += __uint_as_float(raw[n][1][1]);
        }
      }
      const __hip_bfloat16* nw =
          (const __hip_bfloat16*)(u < QPG ? proj.q_norm : proj.k_norm);
      if (nw && u <= QPG) {
        const float inv =
            rsqrtf(wave_sum(x[0] * x[0] + x[1] * x[1]) / DIM + proj.eps);
        x[0] *= inv * bf2f(nw[lane]);
        x[1] *= inv * bf2f(nw[lane + 64]);
      }
      const bool turns = u <= QPG;
      const __hip_bfloat16 o1 = f2bf(turns ? x[0] * co - x[1] * si : x[0]);
      const __hip_bfloat16 o2 = f2bf(turns ? x[1] * co + x[0] * si : x[1]);
      heads_lds[u][lane] = o1;
      heads_lds[u][lane + 64] = o2;
      if (u >= QPG && slot >= 0) {
        __hip_bfloat16* dst = (u == QPG ? keys : values) +
                              (size_t)(slot / PAGE) * page_size + head_at +
                              slot % PAGE * DIM + lane;
        dst[0] = o1;
        dst[64] = o2;
      }
    }
#undef DP_PART
    __syncthreads();
#pragma unroll
    for (int d = 0; d < 4; ++d)
      qf[d] = dp_frag(dp_load(&heads_lds[min(c, QPG - 1)][d * 32 + g * 8]));
    // A step that is asked for from here on has the new row from memory: it stands
    // behind the barrier, and the waves of a workgroup share their CU's cache.
    if (fresh >= 0) {
      const int in = fresh % PAGE;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        // past the last page it is that one: weights of 0 meet its values too
        if (min(at / PAGE + p, last_page) != fresh / PAGE) continue;
#pragma unroll
        for (int d = 0; d < 4; ++d)
          if (in == c) kr[p][d] = dp_load(&heads_lds[QPG][d * 32 + g * 8]);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (in == j * 4 + g) vr[p][j] = dp_load(&heads_lds[QPG + 1][c * 8]);
      }
    }
  }
  for (; at < end; at += WAVES * STEP) {
    const int later[2] = {DP_PAGE(at + 2 * WAVES * STEP, 0),
                          DP_PAGE(at + 2 * WAVES * STEP, 1)};
    f32x4 s[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      s[p] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < 4; ++d)
        s[p] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(dp_frag(kr[p][d]),
                                                       qf[d], s[p], 0, 0, 0);
    }
    DP_KEYS(page)
    __builtin_amdgcn_sched_barrier(0);

    // lane: head c, keys at + 16 p + 4 g + r
    float w[2][4], top = LOW;
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        w[p][r] = at + p * PAGE + g * 4 + r < end ? s[p][r] * scale : LOW;
        top = fmaxf(top, w[p][r]);
      }
    top = fmaxf(top, __shfl_xor(top, 16, 64));
    top = fmaxf(top, __shfl_xor(top, 32, 64));
    const float m_new = fmaxf(m, top);
    const float fade = __builtin_amdgcn_exp2f(m - m_new);
    m = m_new;
    l *= fade;
    union { __hip_bfloat16 e[8]; bf16x8 v; } pf;
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float e = w[p][r] <= LOW
                            ? 0.f : __builtin_amdgcn_exp2f(w[p][r] - m_new);
        l += e;
        pf.e[p * 4 + r] = f2bf(e);
      }
#pragma unroll
    for (int t = 0; t < 8; ++t) acc[t] *= fade;

#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<dp_u4*>(vl + v_put + p * 256 + j * 64) = vr[p][j];
    DP_VALUES(page)
    page[0] = later[0];
    page[1] = later[1];
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const unsigned va = (unsigned)(unsigned long long)(vl + g * 64 + c * 4);
    unsigned long long lo[8], hi[8];
#define DP_READ(t, a, b, off0, off1)                                       \
    "ds_read_b64_tr_b16 " a ", %16 offset:" off0 "\n\t"                    \
    "ds_read_b64_tr_b16 " b ", %16 offset:" off1 "\n\t"
    asm volatile(
        DP_READ(0, "%0", "%1", "0", "512")
        DP_READ(1, "%2", "%3", "1056", "1568")
        DP_READ(2, "%4", "%5", "2112", "2624")
        DP_READ(3, "%6", "%7", "3168", "3680")
        DP_READ(4, "%8", "%9", "4224", "4736")
        DP_READ(5, "%10", "%11", "5280", "5792")
        DP_READ(6, "%12", "%13", "6336", "6848")
        DP_READ(7, "%14", "%15", "7392", "7904")
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(lo[0]), "=&v"(hi[0]), "=&v"(lo[1]), "=&v"(hi[1]),
          "=&v"(lo[2]), "=&v"(hi[2]), "=&v"(lo[3]), "=&v"(hi[3]),
          "=&v"(lo[4]), "=&v"(hi[4]), "=&v"(lo[5]), "=&v"(hi[5]),
          "=&v"(lo[6]), "=&v"(hi[6]), "=&v"(lo[7]), "=&v"(hi[7])
        : "v"(va)
        : "memory");
#undef DP_READ
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      union { unsigned long long u[2]; bf16x8 v; } vf;
      vf.u[0] = lo[t];
      vf.u[1] = hi[t];
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf.v, pf.v, acc[t], 0,
                                                       0, 0);
    }
  }
#undef DP_PAGE
#undef DP_KEYS
#undef DP_VALUES

  // the waves' sums meet in LDS; lane: head c, dims 16 t + 4 g + r
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  __syncthreads();
  float* meet = reinterpret_cast<float*>(&v_lds[0][0]);
  if (c < QPG) {
#pragma unroll
    for (int t = 0; t < 8; ++t)
      *reinterpret_cast<f32x4*>(
          &meet[(wave * QPG + c) * DIM + t * 16 + g * 4]) = acc[t];
    if (g == 0) {
      sums[wave][c][0] = m;
      sums[wave][c][1] = l;
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < QPG * DIM; e += 64 * WAVES) {
    const int h = e / DIM, d = e % DIM;
    float top = LOW;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) top = fmaxf(top, sums[w][h][0]);
    float o = 0.f, total = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float f = __builtin_amdgcn_exp2f(sums[w][h][0] - top);
      o += meet[(w * QPG + h) * DIM + d] * f;
      total += sums[w][h][1] * f;
    }
    const size_t row = (size_t)seq * heads + kvh * QPG + h;
    if (ctx <= span) {        // no keys: 0; NaN stays
      out[row * DIM + d] = f2bf(total == 0.f ? 0.f : o / total);
    } else {
      const size_t at_row = (size_t)split * seqs * heads + row;
      // past the L2, which other XCDs' workgroups do not see
      dp_share(&part_o[at_row * DIM + d], o);
      if (d == 0) {
        dp_share(&part_ml[at_row * 2], top);
        dp_share(&part_ml[at_row * 2 + 1], total);
      }
    }
  }
  if (!tickets || ctx <= span) return;

  // every thread's sums are there before the ticket is
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __shared__ int taken;
  __syncthreads();
  const int parts = min((ctx + span - 1) / span, splits);
  if (threadIdx.x == 0) {
    int* ticket = tickets + (size_t)seq * kv_heads + kvh;
    taken = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
    if (taken == parts - 1)
      __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (taken != parts - 1) return;
  // four dims a thread, the parts in shares that meet in LDS; rounds of 8
  // independent loads
  constexpr int PIECES = QPG * DIM / 4, SHARES = 64 * WAVES / PIECES;
  const int piece = threadIdx.x % PIECES, share = threadIdx.x / PIECES;
  const int h = piece / (DIM / 4), d = piece % (DIM / 4) * 4;
  const size_t row = (size_t)seq * heads + kvh * QPG + h;
  const size_t step = (size_t)seqs * heads;
  float top = LOW, total = 0.f;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  for (int first = share; first < parts; first += 8 * SHARES) {
    float ms[8], ls[8];
    f32x4 os[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      // past the end: the last part again, without weight
      const size_t from = min(first + i * SHARES, parts - 1) * step + row;
      const f32x2 ml = dp_shared(part_ml + from * 2);
      const f32x2 lo = dp_shared(part_o + from * DIM + d);
      const f32x2 hi = dp_shared(part_o + from * DIM + d + 2);
      ms[i] = ml[0];
      ls[i] = ml[1];
      os[i] = f32x4{lo[0], lo[1], hi[0], hi[1]};
    }
    float most = top;
#pragma unroll
    for (int i = 0; i < 8; ++i) most = fmaxf(most, ms[i]);
    const float fade = __builtin_amdgcn_exp2f(top - most);
    top = most;
    o *= fade;
    total *= fade;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (first + i * SHARES < parts) {
        const float f = __builtin_amdgcn_exp2f(ms[i] - top);
        o += os[i] * f;
        total += ls[i] * f;
      }
  }
  if (SHARES > 1) {
    // `meet` was read before the barriers above; [share][piece][o, top, total]
    float* mine = meet + (share * PIECES + piece) * 6;
#pragma unroll
    for (int j = 0; j < 4; ++j) mine[j] = o[j];
    mine[4] = top;
    mine[5] = total;
    __syncthreads();
    if (share) return;
    float most = LOW;
#pragma unroll
    for (int k = 0; k < SHARES; ++k)
      most = fmaxf(most, meet[(k * PIECES + piece) * 6 + 4]);
    o = f32x4{0.f, 0.f, 0.f, 0.f};
    total = 0.f;
#pragma unroll
    for (int k = 0; k < SHARES; ++k) {
      const float* theirs = meet + (k * PIECES + piece) * 6;
      const float f = __builtin_amdgcn_exp2f(theirs[4] - most);
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] += theirs[j] * f;
      total += theirs[5] * f;
    }
  }
  union { __hip_bfloat16 e[4]; uint2 u; } b;
#pragma unroll
  for (int j = 0; j < 4; ++j) b.e[j] = f2bf(total == 0.f ? 0.f : o[j] / total);
  *reinterpret_cast<uint2*>(out + row * DIM + d) = b.u;
}

}  // namespace

// heads_in: null where q is as attention takes it; else q, or its sums, are rows of
// q | k | v heads as the projection left them
extern "C" void launch_decode_pages(
    void* out, void* part_o, void* part_ml, const void* q, void* keys,
    void* values, const void* tables, const void* lens, float scale,
    int seqs, int heads, int kv_heads, int max_pages, int splits, int span,
    int q_stride, void* tickets, const DecodeHeads* heads_in,
    hipStream_t stream) {
  // in whole rounds of the waves
  span = max(1, (span + PART_ROUND - 1) / PART_ROUND) * PART_ROUND;
  // Where pairs of sequence and key head fill the chip three times, no part of a
  // few keys beside one of many (128 sequences of 2080 and 8 heads 181 -> 171 us,
  // 96 of up to 2500 106 -> 101; 64 of up to 4000 143 -> 146, so not for fewer).
  const int whole = seqs * kv_heads >= 768 ? span + span / 4 : span;
  // Up to as many sequences as a key head has CUs, and 64, whose lengths a wave sees
  // at once: workgroups are dealt out by the lengths, one for every CU (comment above).
  // More sequences leave two or three on a CU either way, and no order of parts of 512
  // to 2048 keys was better (45 of up to 2500 60 to 67 us).
  const int cus = 256 / kv_heads;
  const int slots = tickets && splits > 1 && seqs <= min(cus, 64) &&
                            (int64_t)seqs * max_pages < 1 << 23   // even_keys
                        ? min(cus, seqs * splits) : 0;
  // a second one where sequences may use up the first (even_keys); it costs a batch
  // that does not take it up to 0.3 us
  const int most = seqs * 4 <= cus ? 1 : 2;
  const dim3 grid(kv_heads, slots ? min(slots * most, seqs * splits) : seqs,
                  slots ? 1 : splits);
  const dim3 block(64 * WAVES);
#define DP_LAUNCH(QPG, TOGETHER, PROJ)                                     \
  decode_pages_kernel<QPG, TOGETHER, PROJ><<<grid, block, 0, stream>>>(    \
      (const int*)lens, kv_heads, seqs, splits, most, (const int*)tables,  \
      max_pages, span, whole, slots,                                       \
      (const __hip_bfloat16*)q, q_stride,                                  \
      scale * 1.44269504088896f, (__hip_bfloat16*)keys,                    \
      (__hip_bfloat16*)values, (float*)part_o, (float*)part_ml,            \
      (__hip_bfloat16*)out, (int*)tickets,                                 \
      heads_in ? *heads_in : DecodeHeads{})
#define DP_GO(QPG)                                                         \
  do {                                                                     \
    if (seqs >= 96 && heads_in) DP_LAUNCH(QPG, true, true);                \
    else if (seqs >= 96) DP_LAUNCH(QPG, true, false);                      \
    else if (heads_in) DP_LAUNCH(QPG, false, true);                        \
    else DP_LAUNCH(QPG, false, false);                                     \
  } while (0)
  switch (heads / kv_heads) {
    case 1: DP_GO(1); break;
    case 2: DP_GO(2); break;
    case 4: DP_GO(4); break;
    case 8: DP_GO(8); break;
    default: return;        // refused by the caller
  }
#undef DP_LAUNCH
#undef DP_GO
  if (tickets) return;
  // sums to the base of 2
  launch_decode_join((__hip_bfloat16*)out, (const float*)part_o,
                     (const float*)part_ml, (const int*)lens, span, whole,
                     splits, heads, seqs, 1.f, stream);
}
