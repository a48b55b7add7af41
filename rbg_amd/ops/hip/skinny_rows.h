// Decode GEMM of a few rows, C[M,N] = A[M,K] x W[N,K]^T, M <= 4.
#pragma once
#include "common.h"

namespace {

typedef __attribute__((ext_vector_type(4))) unsigned int sg_u4;

DEV_INLINE sg_u4 sg_load(const __hip_bfloat16* p) {
  return *reinterpret_cast<const sg_u4*>(p);
}

DEV_INLINE bf16x8 sg_frag(sg_u4 u) {
  union { sg_u4 u; bf16x8 v; } c;
  c.u = u;
  return c.v;
}

DEV_INLINE float silu(float g) { return g / (1.f + __expf(-g)); }

// The chunk that a workgroup takes as its c-th.
DEV_INLINE int sg_turn(int c, int first, int n) {
  c += first;
  return c >= n ? c - n : c;
}

constexpr int ROWS_KC = 64, ROWS_DEPTH = 4, ROWS_MOST = 4;

// 8 waves share one 16-row tile of W and take its K in turns, without a
// barrier until their sums meet in LDS, and without splits whose sums another
// launch would add.  4096 x 4096, one row: 8.5 us against 10.5 of
// skinny_gemm_kernel with its reduction.  Its time grows with the rows, since
// every workgroup reads all of A (28672 x 4096: 1 row 41.8 us, 4 rows 44.3).
// Where stream_rows.hip is linked it takes what has 1024 columns and k or more, but
// the widest of 2048 k (ops._stream); this takes the others, and all of them in a
// process with an extension of another family alone.
// GLU: W's halves are gate and up, the tile is 8 rows of each: silu(gate) * up.
// PAIR: the tile is 8 rows of W, whose k are taken two chunks at a time, so that
// twice as many workgroups are half as long.  For matrices whose tiles of 16 rows
// leave half of the chip or more idle, with long k (1 row: 1024 x 4096 8.0 -> 6.1
// us, 2048 x 5632 10.6 -> 9.8, x 14336 19.6 -> 15.8, x 2048 6.1 -> 6.5; 4 rows: 2048
// x 4096 8.9 -> 8.4), and where they fill it one and a half times (1 row of 5120 x
// 8192 24.1 -> 19.5, of 6144 x 25600 69 -> 58; 4 rows 25.4 -> 25.1, 74 -> 78).
template <bool GLU, bool PAIR>
__global__ __launch_bounds__(512, 2) void skinny_rows_kernel(
    const __hip_bfloat16* __restrict__ w,   // [N, K]
    const __hip_bfloat16* __restrict__ a,   // [M, K]
    const int K, const int N, const int M,
    __hip_bfloat16* __restrict__ c,         // [M, N], GLU: [M, N / 2]
    float* __restrict__ wide) {             // not null: C in f32, not GLU
  static_assert(!PAIR || !GLU, "plain products only");
  constexpr int WAVES = 8, STEP = PAIR ? 2 * ROWS_KC : ROWS_KC;
  __shared__ __align__(16) float red[WAVES * 16 * ROWS_MOST];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int col0 = blockIdx.x * (PAIR || GLU ? 8 : 16);
  const int row = PAIR ? col0 + (r & 7)
                  : GLU ? col0 + (r & 7) + (r >> 3) * (N / 2) : col0 + r;
  // PAIR: W's second 8 rows and A's second 4 stand for the first ones' next k
  const __hip_bfloat16* wp = w + (size_t)row * K + wave * STEP + g * 8 +
                             (PAIR ? (r >> 3) * ROWS_KC : 0);
  const __hip_bfloat16* ap = a + (size_t)min(PAIR ? r & 3 : r, M - 1) * K +
                             wave * STEP + g * 8 +
                             (PAIR ? (r >> 2 & 1) * ROWS_KC : 0);
  const int n = (K / STEP - wave + WAVES - 1) / WAVES;
  const int first = n ? ((blockIdx.x >> 3) + (blockIdx.x & 7) * (n >> 3)) % n
                      : 0;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  sg_u4 wr[ROWS_DEPTH][2], ar[ROWS_DEPTH][2];
#define SR_WEIGHTS(s, at)                                                  \
  do {                                                                     \
    const int off = sg_turn(at, first, n) * (STEP * WAVES);                \
    wr[s][0] = sg_load(wp + off);                                          \
    wr[s][1] = sg_load(wp + off + 32);                                     \
  } while (0)
#define SR_ROWS(s, at)                                                     \
  do {                                                                     \
    const int off = sg_turn(at, first, n) * (STEP * WAVES);                \
    ar[s][0] = sg_load(ap + off);                                          \
    ar[s][1] = sg_load(ap + off + 32);                                     \
  } while (0)
#define SR_MATH(s)                                                         \
  do {                                                                     \
    _Pragma("unroll") for (int h = 0; h < 2; ++h)                          \
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(                     \
            sg_frag(ar[s][h]), sg_frag(wr[s][h]), acc, 0, 0, 0);           \
  } while (0)
  if (n > 0) {
#pragma unroll
    for (int s = 0; s < ROWS_DEPTH; ++s) SR_WEIGHTS(s, min(s, n - 1));
  }
  if (n > 0) {
#pragma unroll
    for (int s = 0; s < ROWS_DEPTH; ++s) SR_ROWS(s, min(s, n - 1));
    int at = 0;
    for (; at + ROWS_DEPTH < n; at += ROWS_DEPTH) {
#pragma unroll
      for (int s = 0; s < ROWS_DEPTH; ++s) {
        SR_MATH(s);
        SR_WEIGHTS(s, min(at + ROWS_DEPTH + s, n - 1));
        SR_ROWS(s, min(at + ROWS_DEPTH + s, n - 1));
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int s = 0; s < ROWS_DEPTH; ++s)
      if (at + s < n) SR_MATH(s);
  }
#undef SR_WEIGHTS
#undef SR_ROWS
#undef SR_MATH

  // lane l, register q: row 4 * (l >> 4) + q of A, row l & 15 of the tile; only
  // the first ROWS_MOST rows are there, the first 16 lanes'
  if (PAIR ? g == r >> 3 : g == 0)
    *reinterpret_cast<f32x4*>(red + (wave * 16 + r) * ROWS_MOST) = acc;
  __syncthreads();
  const int e = threadIdx.x;
  if (e >= 16 * ROWS_MOST) return;
  const int col = e / ROWS_MOST, m = e % ROWS_MOST;
  if (m >= M || ((PAIR || GLU) && col >= 8)) return;
  float v = 0.f, v2 = 0.f;
#pragma unroll
  for (int k = 0; k < WAVES; ++k) {
    v += red[k * 16 * ROWS_MOST + e];
    if (PAIR || GLU) v2 += red[k * 16 * ROWS_MOST + e + 8 * ROWS_MOST];
  }
  if (PAIR) v += v2;
  if (GLU) c[(size_t)m * (N / 2) + col0 + col] = f2bf(silu(v) * v2);
  else if (wide) wide[(size_t)m * N + col0 + col] = bf2f(f2bf(v));
  else c[(size_t)m * N + col0 + col] = f2bf(v);
}

template <bool GLU, bool PAIR = false>
void launch_skinny_rows(__hip_bfloat16* c, const __hip_bfloat16* a,
                        const __hip_bfloat16* w, int M, int N, int K,
                        hipStream_t stream, float* wide = nullptr) {
  skinny_rows_kernel<GLU, PAIR>
      <<<dim3(N / (PAIR ? 8 : 16)), dim3(512), 0, stream>>>(w, a, K, N, M, c,
                                                           wide);
}

}  // namespace
