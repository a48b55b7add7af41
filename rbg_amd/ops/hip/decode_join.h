// Parts of a sequence in decode attention, and the sum of what they left.
#pragma once
#include "common.h"

namespace {

constexpr int DIM = 128, PART_ROUND = 128;
constexpr float LOW = -1e30f;

// Keys of a part: not a share of the table's capacity, which may be many times
// a sequence's length (one of 2048 keys, 8 heads, tables of 8192 / 40960 /
// 131072 keys: 11.0 / 20.7 / 27.4 us with shares of the capacity, 11.1 of any).
// Up to `whole` keys are one part all the same.
DEV_INLINE int part_keys(int ctx, int least, int whole, int splits) {
  if (ctx > least && ctx <= whole)
    return (ctx + PART_ROUND - 1) / PART_ROUND * PART_ROUND;
  if (ctx <= least * splits) return least;
  const int all = splits * PART_ROUND;
  return (ctx + all - 1) / all * PART_ROUND;
}

// Sums, or the largest, of a lane's value and those of the lanes below; of none 0.
template <bool MAX>
DEV_INLINE int up_to_lane(int x) {
#define DJ_STEP(ctrl, rows)                                                \
  do {                                                                     \
    const int y = __builtin_amdgcn_update_dpp(0, x, ctrl, rows, 0xf, false); \
    x = MAX ? max(x, y) : x + y;                                           \
  } while (0)
  DJ_STEP(0x111, 0xf);            // by 1, 2, 4 and 8 lanes of a row of 16
  DJ_STEP(0x112, 0xf);
  DJ_STEP(0x114, 0xf);
  DJ_STEP(0x118, 0xf);
  DJ_STEP(0x142, 0xa);            // a row's last to the next, 31 to the upper half
  DJ_STEP(0x143, 0xc);
#undef DJ_STEP
  return x;
}

// Rounds of a part below which there is none: up to three are one part; a sequence
// has as many as its join reads at once, `joins`, or 512 keys each (one of 300 / 1000 /
// 2048 / 4000 / 8000 keys, 4 query heads, us: parts of 128 7.8 / 8.1 / 9.1 / 12.2 /
// 19.9, of 256 8.6 / 9.2 / 9.6 / 10.4 / 14.3, of 512 7.1 / 11.7 / 12.2 / 12.2 / 13.1).
DEV_INLINE int least_rounds(int longest, int joins) {
  return longest <= 3 ? 3 : min(4, (longest + joins - 1) / joins);
}

// ceil(x / y), exact for x + y to 2^21 (the quotient of x + y - 1/2 is 1/(2y) away from whole
// numbers, and off by 2^-22 of itself at most): a division of whole numbers is 0.15 us
// of a search for parts, which has several.
DEV_INLINE int over(int x, int y) {
  return (int)(((float)(x + y) - 0.5f) * __builtin_amdgcn_rcpf((float)y));
}

// Keys of a part where the sequences of a batch, at most 64, share `slots`
// workgroups a key head: as few as leave none over, or a sixteenth more, but not below
// the above, nor so few that a sequence has more than `splits` parts.  Sequences that
// use up the slots, and rows that stand for none, leave no cut for a long one: two
// workgroups a slot then (`most`), if that saves more than a fifth of the keys of a
// slot; a CU whose others have ended reads up to 2.5 times faster, so that less is no
// gain (8 key heads, us, one a slot / two: 31 of 500 and one of 16000 181 / 42, 17 of
// 8000 in 24 rows 119 / 105, 9 of 15000 in 16 118 / 101, 20 of 400 to 6000 in 24 63 /
// 59, 32 of 200 to 2500 42 / 44, 24 of 8000 131 / 153; with three a slot as with two, to
// 2%).  n: lane i has the length of sequence i, others 0.  `parts` are the lane's, one
// where it has no keys, and `upto` those of all sequences to it.
DEV_INLINE int even_keys(const int n, const int seqs, const int slots,
                         const int most, const int joins, const int splits,
                         int* parts, int* upto) {
  const int lane = threadIdx.x & 63;
  const int rounds = (max(n, 0) + PART_ROUND - 1) / PART_ROUND;
  const int longest = __builtin_amdgcn_readlane(up_to_lane<true>(rounds), 63);
  const int least = least_rounds(longest, joins);
  *parts = lane < seqs;
  *upto = min(lane + 1, seqs);
  if (longest <= least) return least * PART_ROUND;
  const int all = __builtin_amdgcn_readlane(up_to_lane<false>(rounds), 63);
  const int from = max(least, over(longest, splits));
  const auto fit = [&](int span, int places) {
    *parts = lane < seqs ? max(1, over(rounds, span)) : 0;
    *upto = up_to_lane<false>(*parts);
    return __builtin_amdgcn_readlane(*upto, 63) <= places;
  };
  const auto shortest = [&](int places) {
    int low = max(from, over(all, places));
    if (fit(low, places)) return low;
    // a sequence has less than one part above its share
    int high = places > seqs ? min(longest, over(all, places - seqs)) : longest;
    while (high - low > max(1, low / 16)) {
      const int mid = (low + high) / 2;
      if (fit(mid, places)) high = mid;
      else low = mid;
    }
    fit(high, places);
    return high;
  };
  int span = shortest(slots);
  if (most > 1 && span * slots > all + all / 2) {
    const int two = shortest(2 * slots);
    if (two * 5 < span * 2) span = two;
    else fit(span, slots);
  }
  return span * PART_ROUND;
}

// The same of one sequence.
DEV_INLINE int even_keys(const int ctx, const int slots, const int joins,
                         const int splits) {
  const int rounds = (max(ctx, 0) + PART_ROUND - 1) / PART_ROUND;
  const int most = min(slots, splits);
  return max(least_rounds(rounds, joins), (rounds + most - 1) / most) *
         PART_ROUND;
}

// A workgroup per query head adds the parts' sums, in shares that meet in LDS.
// Bound by latency: the loads of a round of 8 parts are independent (one load
// after another took 9-10 us for 16 parts of one sequence).  Of more than 8
// parts there are four shares (3 sequences of up to 15000 tokens, 30 parts: 40.7
// -> 36.7 us with the attention); else one, whose workgroups are a quarter of
// the threads (128 x 2080: 174 us against 180).
// lens: parts are of part_keys(length, least, whole, splits), a sequence of one part
// has no sums.  null: every sequence has `splits` of them, perhaps empty ones.
// to_base2: of the maxima, 1 or log2(e).
template <int SHARES>
__global__ __launch_bounds__(DIM * SHARES) void decode_join_kernel(
    __hip_bfloat16* __restrict__ out,       // [seqs, QH, DIM]
    const float* __restrict__ part_o,       // [splits, seqs, QH, DIM]
    const float* __restrict__ part_ml,      // [splits, seqs, QH, 2]
    const int* __restrict__ lens, const int least, const int whole,
    const int splits, const float to_base2) {
  const int seq = blockIdx.y, d = threadIdx.x % DIM;
  const int share = threadIdx.x / DIM;
  int n = splits;
  if (lens) {
    const int ctx = lens[seq], span = part_keys(ctx, least, whole, splits);
    if (ctx <= span) return;
    n = min((ctx + span - 1) / span, splits);
  }
  const size_t row = (size_t)seq * gridDim.x + blockIdx.x;
  const size_t step = (size_t)gridDim.y * gridDim.x;
  __shared__ float meet[SHARES][DIM + 2];
  float top = LOW, o = 0.f, total = 0.f;
  for (int first = share; first < n; first += 8 * SHARES) {
    float ms[8], ls[8], os[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      // past the end: the last part again, without weight
      const size_t at = min(first + i * SHARES, n - 1) * step + row;
      ms[i] = part_ml[at * 2] * to_base2;
      ls[i] = part_ml[at * 2 + 1];
      os[i] = part_o[at * DIM + d];
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
      if (first + i * SHARES < n) {
        const float f = __builtin_amdgcn_exp2f(ms[i] - top);
        o += os[i] * f;
        total += ls[i] * f;
      }
  }
  meet[share][d] = o;
  if (d == 0) {
    meet[share][DIM] = top;
    meet[share][DIM + 1] = total;
  }
  __syncthreads();
  if (share) return;
#pragma unroll
  for (int k = 0; k < SHARES; ++k) top = fmaxf(top, meet[k][DIM]);
  o = total = 0.f;
#pragma unroll
  for (int k = 0; k < SHARES; ++k) {
    const float f = __builtin_amdgcn_exp2f(meet[k][DIM] - top);
    o += meet[k][d] * f;
    total += meet[k][DIM + 1] * f;
  }
  // no keys: 0; weights that are no numbers: no number
  out[row * DIM + d] = f2bf(total == 0.f ? 0.f : o / total);
}

inline void launch_decode_join(__hip_bfloat16* out, const float* part_o,
                               const float* part_ml, const int* lens,
                               int least, int whole, int splits, int heads,
                               int seqs, float to_base2, hipStream_t stream) {
  if (splits <= 1) return;
  const dim3 grid(heads, seqs);
  if (splits <= 8)
    decode_join_kernel<1><<<grid, dim3(DIM), 0, stream>>>(
        out, part_o, part_ml, lens, least, whole, splits, to_base2);
  else
    decode_join_kernel<4><<<grid, dim3(DIM * 4), 0, stream>>>(
        out, part_o, part_ml, lens, least, whole, splits, to_base2);
}

}  // namespace
