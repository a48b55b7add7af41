// GEMM of up to 4 rows, C[M,N] = A[M,K] x W[N,K]^T, and the same with the RMS norm
// that makes A and the silu behind the product: the layers of a decode step of one to
// four sequences.
//
// Bound: the weights, read once.  A loop that only reads takes 7.0 us for 4096 x 4096 in
// a graph, 9.6 for 6144 x 4096 and 38.6 for 28672 x 4096 (6.1 TB/s), 1.4 of them from
// launch to launch.  What it took to come near that, against the tiles of 16 rows of W
// before (1 row, norm and silu included):
//  * Order of reading.  A wave has an eighth of K, for all rows of its workgroup, and a
//    load brings 1 KB of a row: a workgroup reads its rows from end to end.  Waves that
//    take K in turns of 64 or 128 for 16 rows, 64 bytes of each in a load, read 6144 x
//    4096 in 13.2 us.
//  * Operands.  16 bytes of one row of W are the operands of v_mfma_f32_4x4x4, 16 blocks
//    of 4 rows of W, 4 rows of A and 4 k, when a lane of four has each row; they turn
//    around on the way through LDS of the wave's own, which costs nothing here.  Sums
//    of the blocks are added once a group, by exchanges of lanes.
//  * Work of a workgroup: little, so that the chip's 256 CUs share the weights evenly
//    and many waves wait at a time, but for the norm that each does for itself.
//  * The norm.  A wave needs only its own k of A: it loads them before its weights and
//    keeps them in registers, without a barrier; the row's 1 / rms, which needs all
//    waves, is a factor of the result.
// 6144 x 4096 12.9 -> 10.5 us, 4 rows 14.6 -> 11.8; 28672 x 4096 with silu 43.4 -> 38.9;
// 51200 x 5120 101 -> 86; 4096 x 4096 without a norm 9.1 -> 7.8; 32768 x 4096 47.5 ->
// 43.7.
#include <algorithm>
#include <type_traits>
#include <utility>

#include "skinny_rows.h"

namespace {

constexpr int SW_SEG = 128, SW_EARLY = 4;

DEV_INLINE f32x4 sw_mfma(sg_u4 a, sg_u4 w, f32x4 acc) {
  union { sg_u4 u; short4_t s[2]; } x, y;
  x.u = a;
  y.u = w;
#pragma unroll
  for (int h = 0; h < 2; ++h)
    acc = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(x.s[h], y.s[h], acc, 0, 0, 0);
  return acc;
}

#define SW_DPP(x, ctrl)                                                    \
  __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(                   \
      0, __builtin_bit_cast(int, x), ctrl, 0xf, 0xf, false))
// The sum of a lane's value over the blocks of its 16 lanes.
DEV_INLINE float sw_row_sum(float x) {
  x += SW_DPP(x, 0x128);        // of those 8 and 4 lanes on
  return x + SW_DPP(x, 0x124);
}

// Sums of the 16 blocks' products: lane l has row l / 16 of A's four and row l % 4 of
// W's.  Halves of the lanes, then of the halves, change what they do not keep.
DEV_INLINE float sw_gather(f32x4 v) {
  float x[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const auto s = __builtin_amdgcn_permlane32_swap(
        __float_as_uint(v[h]), __float_as_uint(v[h + 2]), false, false);
    x[h] = __uint_as_float(s[0]) + __uint_as_float(s[1]);
  }
  const auto s = __builtin_amdgcn_permlane16_swap(
      __float_as_uint(x[0]), __float_as_uint(x[1]), false, false);
  return sw_row_sum(__uint_as_float(s[0]) + __uint_as_float(s[1]));
}

DEV_INLINE sg_u4 sw_load(const char* base, uint32_t off) {
  return *reinterpret_cast<const sg_u4*>(base + off);
}

// What a wave loads of 4 rows of W, SEG segments of 128 k of each: load l brings 64
// pieces of 16 bytes from where the one before ended, row after row, so that a load is
// of one or two rows.  Operands are pieces of all 4 rows: they turn around in LDS of the
// wave's own, pieces exchanged by the row so that nothing conflicts.
template <int SEG>
struct Turn {
  static constexpr int PIECES = SEG * 16, BYTES = 4 * PIECES * 16;
  uint32_t off[SEG];            // bytes from the first row's first segment
  uint32_t put[SEG];
  uint32_t get;
  // segs: how many of the segments there are; the others are the last once more
  DEV_INLINE Turn(int lane, int K, int segs) {
#pragma unroll
    for (int l = 0; l < SEG; ++l) {
      const int p = l * 64 + lane, row = p / PIECES, at = p % PIECES;
      off[l] = (uint32_t)(row * K * 2 +
                          (at < segs * 16 ? at : segs * 16 - 16 + (at & 15)) * 16);
      put[l] = (uint32_t)((row * PIECES + (at ^ (row * 4))) * 16);
    }
    get = (uint32_t)(((lane & 3) * PIECES + ((lane >> 2) ^ ((lane & 3) * 4))) * 16);
  }
  DEV_INLINE void around(char* lds, const sg_u4 (&in)[SEG],
                         sg_u4 (&out)[SEG]) const {
#pragma unroll
    for (int l = 0; l < SEG; ++l) *reinterpret_cast<sg_u4*>(lds + put[l]) = in[l];
    meet();
#pragma unroll
    for (int s = 0; s < SEG; ++s)
      out[s] = *reinterpret_cast<const sg_u4*>(lds + get + s * 256);
    meet();                       // the next turn's stores stay behind these loads
  }
  // What lanes stored is there for the others of the wave: no instruction, but a bound
  // on the compiler's order (644 shapes 0.99 to 1.0 of the time without; 12288 x 7168
  // with a norm, 1 row 34.3 -> 31.0 us, 4096 x 7168, 4 rows 14.7 -> 15.1).
  DEV_INLINE static void meet() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
  }
};

// The waves' sums of `held` groups of rows of W, [waves][row][4], added up and stored
// for this workgroup's units from u0 on: in c, or in f32, rounded to bf16 or not, in
// wide.  squares: [waves][4], of the rows' norms.
template <bool GLU, int WAVES>
DEV_INLINE void sw_store(const float* red, int held, int units, int u0, int M,
                         int N, const float* squares, int K, float eps,
                         __hip_bfloat16* __restrict__ c, float* wide,
                         bool round) {
  const int cols = units * 4, step = held * 16;
  for (int e = threadIdx.x; e < cols * M; e += 64 * WAVES) {
    const int m = e / cols, col = e - m * cols;
    const float* at = red + (GLU ? col / 4 * 8 + col % 4 : col) * 4 + m;
    float v = 0.f, v2 = 0.f, total = 0.f;
#pragma unroll
    for (int k = 0; k < WAVES; ++k) {
      v += at[k * step];
      if (GLU) v2 += at[k * step + 16];
      if (squares) total += squares[k * 4 + m];
    }
    if (squares) {
      const float factor = rsqrtf(total / K + eps);
      v *= factor;
      v2 *= factor;
    }
    if (GLU) c[(size_t)m * (N / 2) + u0 * 4 + col] = f2bf(silu(v) * v2);
    else if (wide) wide[(size_t)m * N + u0 * 4 + col] = round ? bf2f(f2bf(v)) : v;
    else c[(size_t)m * N + u0 * 4 + col] = f2bf(v);
  }
}

// A lane's value of lane q of its four.
template <int Q>
DEV_INLINE sg_u4 sw_quad(sg_u4 v) {
#pragma unroll
  for (int j = 0; j < 4; ++j)
    v[j] = __builtin_amdgcn_update_dpp(0, (int)v[j], Q * 0x55, 0xf, 0xf, false);
  return v;
}

// f of 0 .. N - 1 as constants
template <class F, int... I>
DEV_INLINE void sw_each_of(F f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>()), ...);
}
template <int N, class F>
DEV_INLINE void sw_each(F f) {
  sw_each_of(f, std::make_integer_sequence<int, N>());
}

// A: the RMS norm of src + residual, M <= ROWS rows; src in bf16 or (SUMS) f32.  SEG: most segments of 128 k that a
// wave has.  GD: groups of 4 rows of W asked for ahead.  GLU: W's halves are gate and up;
// a unit is a group of each, else one group.
template <bool GLU, bool SUMS, int ROWS, int WAVES, int SEG, int GD>
__global__ __launch_bounds__(64 * WAVES, WAVES / 4) void norm_stream_kernel(
    const __hip_bfloat16* __restrict__ w,         // [N, K]
    const int K, const int N, const int base, const int extra,
    const void* __restrict__ src,                 // [M, K] or null
    const __hip_bfloat16* __restrict__ residual,  // [M, K]
    const __hip_bfloat16* __restrict__ norm_weight, const int M,
    const float eps, __hip_bfloat16* __restrict__ residual_out,
    __hip_bfloat16* __restrict__ c,               // [M, N], GLU: [M, N / 2]
    float* __restrict__ wide) {                   // not null: C in f32
  extern __shared__ __align__(16) char sw_lds[];
  float* sw_red = (float*)(sw_lds + WAVES * Turn<SEG>::BYTES);
  __shared__ float squares[WAVES][4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 3, b = lane >> 2;
  const int bid = blockIdx.x;
  const int units = base + (bid < extra), u0 = bid * base + min(bid, extra);
  const int groups = GLU ? 2 * units : units;
  const int s0 = K / SW_SEG * wave / WAVES;
  const int segs = K / SW_SEG * (wave + 1) / WAVES - s0;

  // This wave's k of the rows that become A, asked for first: they are few.  A load is
  // of a segment of four rows, as the operands are; of fewer rows it is of four (row,
  // segment) pairs in order, and operands are handed around.
  constexpr bool DIRECT = ROWS == 4;
  constexpr int PAIRS = ROWS * SEG, LOADS = (PAIRS + 3) / 4;
  sg_u4 xs[LOADS][SUMS ? 2 : 1], rs[LOADS], nw[LOADS];
  auto pair_row = [&](int l) {
    return DIRECT ? i : min(l * 4 + i, PAIRS - 1) / SEG;
  };
  auto pair_seg = [&](int l) {
    return DIRECT ? l : min(l * 4 + i, PAIRS - 1) % SEG;
  };
#pragma unroll
  for (int l = 0; l < LOADS; ++l) {
    const int k = (s0 + min(pair_seg(l), segs - 1)) * SW_SEG + b * 8;
    const size_t at = (size_t)min(pair_row(l), M - 1) * K + k;
    rs[l] = sg_load(residual + at);
    // without src the residual stands for it, to no use: a branch costs registers
    if (SUMS) {
      const sg_u4* from = (const sg_u4*)((const float*)src + at);
      xs[l][0] = from[0];
      xs[l][SUMS ? 1 : 0] = from[1];
    } else {
      xs[l][0] =
          sg_load((src ? (const __hip_bfloat16*)src : residual) + at);
    }
    nw[l] = sg_load(norm_weight + k);
  }
  __builtin_amdgcn_sched_barrier(0);

  const char* wb = (const char*)(w + (size_t)u0 * 4 * K + s0 * SW_SEG);
  const Turn<SEG> turn(lane, K, segs);
  char* mine = (char*)sw_lds + wave * Turn<SEG>::BYTES;
  sg_u4 wr[GD][SEG];
  auto weights = [&](int d, int q) {
    const char* p = wb + (size_t)(GLU ? q >> 1 : q) * (4 * 2 * (size_t)K) +
                    (GLU && (q & 1) ? (size_t)N * K : 0);   // 2 N / 2 K
#pragma unroll
    for (int s = 0; s < SEG; ++s) wr[d][s] = sw_load(p, turn.off[s]);
  };
  // some weights before the norm's arithmetic, which they cover, but no more: a wave
  // waits until what it asks for is taken
  constexpr int EARLY = std::min(GD, std::max(1, SW_EARLY / SEG));
#pragma unroll
  for (int d = 0; d < EARLY; ++d) weights(d, min(d, groups - 1));
  __builtin_amdgcn_sched_barrier(0);

  sg_u4 normed[LOADS], ar[SEG];
  float ss[ROWS] = {};          // DIRECT: of row i, in the first
#pragma unroll
  for (int l = 0; l < LOADS; ++l) {
    union U { sg_u4 u; __hip_bfloat16 e[8]; } x, r, g, o;
    x.u = xs[l][0] & (src ? ~0u : 0u);
    r.u = rs[l];
    g.u = nw[l];
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float v = (SUMS ? __uint_as_float(xs[l][SUMS ? j >> 2 : 0][j & 3])
                            : bf2f(x.e[j])) + bf2f(r.e[j]);
      sum += v * v;
      r.e[j] = f2bf(v);
    }
    rs[l] = r.u;
    const bool live = l * 4 + i < PAIRS && pair_seg(l) < segs;
#pragma unroll
    for (int j = 0; j < 8; ++j) o.e[j] = f2bf(bf2f(r.e[j]) * bf2f(g.e[j]));
    normed[l] = live ? o.u : sg_u4{0, 0, 0, 0};
    if (DIRECT) {
      ss[0] += live ? sum : 0.f;
    } else {
#pragma unroll
      for (int m = 0; m < ROWS; ++m)
        ss[m] += live && pair_row(l) == m ? sum : 0.f;
    }
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int d = EARLY; d < GD; ++d) weights(d, min(d, groups - 1));
  __builtin_amdgcn_sched_barrier(0);
  // the operand of segment s: lane i of four has row i
  sw_each<SEG>([&](auto seg) {
    constexpr int s = decltype(seg)::value;
    if constexpr (DIRECT) {
      ar[s] = normed[s];
    } else {
      sw_each<ROWS>([&](auto row) {
        constexpr int m = decltype(row)::value, p = m * SEG + s;
        const sg_u4 v = sw_quad<p % 4>(normed[p / 4]);
        ar[s] = m == 0 || i == m ? v : ar[s];
      });
    }
  });
  if (src && bid == 0) {
#pragma unroll
    for (int l = 0; l < LOADS; ++l)
      if (l * 4 + i < PAIRS && pair_seg(l) < segs && pair_row(l) < M)
        *reinterpret_cast<sg_u4*>(residual_out + (size_t)pair_row(l) * K +
                                  (s0 + pair_seg(l)) * SW_SEG + b * 8) = rs[l];
  }
  if (DIRECT) {
    float v = sw_row_sum(ss[0]);
    v += __shfl_xor(v, 16, 64);
    v += __shfl_xor(v, 32, 64);
    if (lane < 4) squares[wave][lane] = v;
  } else {
#pragma unroll
    for (int m = 0; m < ROWS; ++m) {
      const float v = wave_sum(ss[m]);
      if (lane == 0) squares[wave][m] = v;
    }
  }

  float* red = sw_red + (size_t)wave * groups * 16;
  auto group = [&](int d, int q) {
    sg_u4 wf[SEG];
    turn.around(mine, wr[d], wf);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < SEG; ++s)           // waves differ by a segment at most
      if (s < SEG - 1 || segs == SEG) acc = sw_mfma(ar[s], wf[s], acc);
    const float v = sw_gather(acc);
    if ((lane & 12) == 0) red[(q * 4 + i) * 4 + (lane >> 4)] = v;
  };
  int q = 0;
  for (; q + GD < groups; q += GD) {
#pragma unroll
    for (int d = 0; d < GD; ++d) {
      group(d, q + d);
      weights(d, min(q + d + GD, groups - 1));
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int d = 0; d < GD; ++d)
    if (q + d < groups) group(d, q + d);
  __syncthreads();
  sw_store<GLU, WAVES>(sw_red, groups, units, u0, M, N, &squares[0][0], K, eps, c,
                       wide, false);
}

// A as it is, of any length, M <= 4 rows: G groups of 4 rows of W, GLU: of gate and of
// up in turns.  A turn is SEG segments of 128 k; the next is asked for as this one's
// registers are used.
template <bool GLU, int SEG, int G>
__global__ __launch_bounds__(512, 2) void stream_kernel(
    const __hip_bfloat16* __restrict__ w,         // [N, K]
    const int K, const int N, const __hip_bfloat16* __restrict__ a, // [M, K]
    const int M, __hip_bfloat16* __restrict__ c,  // [M, N], GLU: [M, N / 2]
    float* __restrict__ wide,                     // not null: C in f32
    const bool round) {                           // to bf16 all the same
  extern __shared__ __align__(16) char sw_lds[];
  float* sw_red = (float*)(sw_lds + 8 * Turn<SEG>::BYTES);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 3, b = lane >> 2;
  constexpr int UNITS = GLU ? G / 2 : G;
  const int u0 = blockIdx.x * UNITS;
  const int units = min(UNITS, N / (GLU ? 8 : 4) - u0);
  constexpr int K_TURN = SEG * SW_SEG;
  const int t0 = K / K_TURN * wave / 8;
  const int n = K / K_TURN * (wave + 1) / 8 - t0;
  const char* wb = (const char*)(w + (size_t)u0 * 4 * K + t0 * K_TURN);
  const char* ab = (const char*)(a + t0 * K_TURN);
  const Turn<SEG> turn(lane, K, SEG);
  char* mine = (char*)sw_lds + wave * Turn<SEG>::BYTES;
  const uint32_t ao = (uint32_t)(min(i, M - 1) * K + b * 8) * 2;
  sg_u4 wr[G][SEG], ar[SEG];
  auto rows = [&](int at) {
#pragma unroll
    for (int s = 0; s < SEG; ++s)
      ar[s] = sw_load(ab + (at * SEG + s) * (SW_SEG * 2), ao);
  };
  auto weights = [&](int g, int at) {
    const char* p = wb +
                    (size_t)min(GLU ? g / 2 : g, units - 1) * (8 * (size_t)K) +
                    (GLU && g % 2 ? (size_t)N * K : 0) + at * (K_TURN * 2);
#pragma unroll
    for (int s = 0; s < SEG; ++s) wr[g][s] = sw_load(p, turn.off[s]);
  };
  f32x4 acc[G];
#pragma unroll
  for (int g = 0; g < G; ++g) acc[g] = {0.f, 0.f, 0.f, 0.f};
  auto math = [&](int g) {
    sg_u4 wf[SEG];
    turn.around(mine, wr[g], wf);
#pragma unroll
    for (int s = 0; s < SEG; ++s) acc[g] = sw_mfma(ar[s], wf[s], acc[g]);
  };
  if (n > 0) {
    rows(0);
#pragma unroll
    for (int g = 0; g < G; ++g) weights(g, 0);
    int at = 0;
    for (; at + 1 < n; ++at) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        math(g);
        weights(g, min(at + 1, n - 1));
        __builtin_amdgcn_sched_barrier(0);
      }
      rows(min(at + 1, n - 1));
      __builtin_amdgcn_sched_barrier(0);
    }
    if (at < n)
#pragma unroll
      for (int g = 0; g < G; ++g) math(g);
  }
  float* red = sw_red + wave * G * 16;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const float v = sw_gather(acc[g]);
    if ((lane & 12) == 0) red[(g * 4 + i) * 4 + (lane >> 4)] = v;
  }
  __syncthreads();
  sw_store<GLU, 8>(sw_red, G, units, u0, M, N, nullptr, K, 0.f, c, wide, round);
}

// Groups asked for ahead, and (below) workgroups.  Of one row the norm is little and
// many workgroups are better, of more rows few (10240 x 8192, 1280 / 256, us: 1 row 29.6
// / 30.4, 4 rows 39.1 / 31.5; with silu 28672 x 4096, 3584 / 1792 / 896 / 256: 1 row 38.9
// / 40.0 / 40.7 / 41.3, 2 rows 43.1 / 40.0 / 41.4 / 41.3, 4 rows - / 42.1 / 42.0 / 42.1).
// Of one row and few k two groups ahead, but where a workgroup has no more than two (us,
// one / two: 3072 x 1024 4.5 / 4.0, x 2048 5.3 / 5.0, but 4096 x 2048 5.6 / 5.8), of many
// k one (8192 x 6144 19.3 / 21.3, 4 rows 21.7 / 21.2; 51200 x 5632 with silu, 2 rows 108
// / 102).
constexpr int norm_stream_ahead(bool glu, int rows, int waves, int seg, bool many) {
  if (glu && rows == 1) return waves == 16 || seg > 4 ? 2 : 1;
  if (waves == 16) return seg < 4 && (glu || rows > 1) ? 2 : 1;
  if (glu) return seg <= 4 ? 2 : 1;
  if (rows == 1) return seg <= 2 && many ? 1 : 2;
  return seg <= 2 ? 4 : seg == 3 ? 3 : 2;
}

int norm_stream_workgroups(bool glu, int rows, int units) {
  int wgs = 256;
  if (glu) wgs = std::max(wgs, (units + rows - 1) / rows);
  else if (rows == 1 && units > 768) wgs = (units + 1) / 2;
  wgs = std::max(wgs, (units + 63) / 64);   // 64 groups' sums in LDS
  return std::min(wgs, units);
}

template <bool GLU, bool SUMS, int ROWS, int WAVES, int SEG>
bool launch_norm_stream(__hip_bfloat16* c, float* wide, const void* src,
                        const __hip_bfloat16* w, int M, int N, int K,
                        const __hip_bfloat16* residual,
                        const __hip_bfloat16* norm_weight, float eps,
                        __hip_bfloat16* residual_out, hipStream_t stream) {
  const int units = N / (GLU ? 8 : 4);
  const int wgs = norm_stream_workgroups(GLU, ROWS, units);
  const int groups = (units + wgs - 1) / wgs * (GLU ? 2 : 1);
  const int lds =
      WAVES * (Turn<SEG>::BYTES + groups * 16 * (int)sizeof(float));
  const auto kernel =
      units > 768
          ? norm_stream_kernel<GLU, SUMS, ROWS, WAVES, SEG,
                               norm_stream_ahead(GLU, ROWS, WAVES, SEG, true)>
          : norm_stream_kernel<GLU, SUMS, ROWS, WAVES, SEG,
                               norm_stream_ahead(GLU, ROWS, WAVES, SEG, false)>;
  if (lds > 64 * 1024 &&
      hipFuncSetAttribute((const void*)kernel,
                          hipFuncAttributeMaxDynamicSharedMemorySize,
                          lds) != hipSuccess)
    return false;
  kernel<<<dim3(wgs), dim3(64 * WAVES), lds, stream>>>(
      w, K, N, units / wgs, units % wgs, src, residual, norm_weight, M, eps,
      residual_out, c, wide);
  return true;
}

}  // namespace

// A: the RMS norm of src + residual, which goes to residual_out; src is bf16 or (sums)
// f32, or null, and nothing goes there then.  C in c, or in f32, not rounded, in wide.
// With glu W's halves are gate and up and C is silu(gate) * up, [M, N / 2].  M <= 4, N of
// 4 (glu: 8), K of 128 from 1024 to 8192.  False: not these, nor gate and up of more rows
// than a launch of the norm's own repays: of sums (which are twice as much to read for
// every workgroup; 51200 x 5120, 2 rows 107 us, so 90), of 3 and 4 rows of more than 4096
// (51200 x 5120 96 / 92, 57344 x 8192 164 / 155).
extern "C" bool launch_norm_rows(void* c, void* wide, const void* src, int sums,
                                 const void* residual, void* residual_out,
                                 const void* norm_weight, float eps,
                                 const void* w, int M, int N, int K, int glu,
                                 hipStream_t stream) {
  if (M < 1 || M > 4 || N < 1 || N % (glu ? 8 : 4) || K % SW_SEG || K < 1024 ||
      K > 8192 || (sums && !src) || (glu && (wide || (sums && M > 1) || (M > 2 && K > 4096))))
    return false;
  const int waves = K > 5120 ? 16 : 8;      // a wave has 5 segments at most
  const int segs = (K / SW_SEG + waves - 1) / waves;
#define SW_FORM(GLU, SUMS, ROWS, WAVES, SEG)                               \
  if ((glu != 0) == GLU && (sums != 0) == SUMS && M <= ROWS &&             \
      waves == WAVES && segs == SEG)                                       \
    return launch_norm_stream<GLU, SUMS, ROWS, WAVES, SEG>(                \
        (__hip_bfloat16*)c, (float*)wide, src, (const __hip_bfloat16*)w, M, \
        N, K, (const __hip_bfloat16*)residual,                             \
        (const __hip_bfloat16*)norm_weight, eps,                           \
        (__hip_bfloat16*)residual_out, stream);
#define SW_ROWS(WAVES, SEG)                                                \
  SW_FORM(true, false, 1, WAVES, SEG) SW_FORM(true, true, 1, WAVES, SEG)   \
  SW_FORM(true, false, 2, WAVES, SEG)                                      \
  SW_FORM(false, false, 1, WAVES, SEG) SW_FORM(false, true, 1, WAVES, SEG) \
  SW_FORM(false, false, 2, WAVES, SEG) SW_FORM(false, true, 2, WAVES, SEG) \
  SW_FORM(false, false, 4, WAVES, SEG) SW_FORM(false, true, 4, WAVES, SEG)
  SW_ROWS(8, 1) SW_ROWS(8, 2) SW_ROWS(8, 3) SW_ROWS(8, 4) SW_ROWS(8, 5)
  SW_ROWS(16, 3) SW_ROWS(16, 4)
  SW_FORM(true, false, 4, 8, 1) SW_FORM(true, false, 4, 8, 2)
  SW_FORM(true, false, 4, 8, 3) SW_FORM(true, false, 4, 8, 4)
#undef SW_ROWS
#undef SW_FORM
  return false;
}

// C in bf16 in c, or, where wide is not null, there in f32, rounded to bf16 or not; with
// glu silu(gate) * up in c.  M <= 4, N of 4, glu: 8, K of 256.  Turns of 512 k where rows
// are long, or many and not short (us, turns of 256 / 512: 5120 x 25600 53.2 / 51.4,
// 32768 x 4096 47.0 / 43.7, x 2048 23.7 / 25.6; 8192 x 5120 15.7 / 16.0).
extern "C" bool launch_stream_rows(void* c, void* wide, int round, const void* a,
                                   const void* w, int M, int N, int K, int glu,
                                   hipStream_t stream) {
  if (M < 1 || M > 4 || N < 1 || N % (glu ? 8 : 4) || K < 256 || K % 256 ||
      (glu && wide))
    return false;
  const bool longer =
      K % 512 == 0 && (K >= 16384 || (N >= 16384 && K >= 4096));
  const auto go = [&](auto kernel, int groups, int seg) {
    // 4 rows of a turn for each of the waves, and their sums
    const int lds = 8 * (seg * 1024 + groups * 16 * (int)sizeof(float));
    kernel<<<dim3((N / 4 + groups - 1) / groups), dim3(512), lds, stream>>>(
        (const __hip_bfloat16*)w, K, N, (const __hip_bfloat16*)a, M,
        (__hip_bfloat16*)c, (float*)wide, round != 0);
  };
  // of narrow matrices a group is enough for a workgroup (1024 x 2048 3.1 / 3.0 us)
  if (glu && longer) go(stream_kernel<true, 4, 2>, 2, 4);
  else if (glu) go(stream_kernel<true, 2, 2>, 2, 2);
  else if (longer) go(stream_kernel<false, 4, 2>, 2, 4);
  else if (N <= 1024) go(stream_kernel<false, 2, 1>, 1, 2);
  else go(stream_kernel<false, 2, 2>, 2, 2);
  return true;
}
