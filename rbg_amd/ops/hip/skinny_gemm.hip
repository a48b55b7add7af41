// Decode-shape GEMM: C[M,N] = A[M,K] x W[N,K]^T, bf16 in, f32 accumulators,
// bf16 out, M <= 256 rows.  Optionally W's two halves are a gate and an up
// matrix and C[M,N/2] = silu(A Wg^T) * (A Wu^T).
//
// Bound: the weights, read once from HBM.  A plain read reaches 6.1-6.3 TB/s
// here, so 28672 x 4096 takes 38 us at best; up to 16 rows take 38 of them,
// 64 take 41 and 128 take 58, whose A panels pass the L2s as often as the
// weights do.
//
// A lane of v_mfma_f32_16x16x32_bf16 holds 8 consecutive k of one row, and the
// lanes beside it other rows.  Loads in that order touch 16 lines for every 16
// lanes, which a CU does at 27 bytes a ns where 256 neighbouring bytes of a row
// give 38, so up to 96 rows a wave loads its chunk as 256 bytes of 4 rows at a
// time and turns it through 4 KB of LDS of its own, without a barrier (28672 x
// 4096: 7 rows of 24576 36.3 -> 33.9 us, 45 rows 43.1 -> 40.3, 64 rows 44.8 ->
// 40.7; 5120 x 25600 in 6 parts, 64 rows 54.9 -> 50.0, 96 rows 62.0 -> 56.3;
// 10240 x 5120 25.2 -> 23.0).  With 128 rows LDS is as busy as the loads, and
// the turn gains nothing (4096 x 4096 in 8: 14.8, turned 15.2).
// What else made the difference, at 28672 x 4096:
//  * plain loads, not non-temporal ones, which send both halves of a line to
//    L2 and back as requests of their own (16 rows: 48 -> 42 us),
//  * loads pinned where they are issued: the compiler otherwise moves A's to
//    their use, behind the MFMAs, and every chunk pays their latency (128
//    rows: 75 -> 64 us),
//  * two lines of a row at a time, not one (57344 x 8192, 1 row: 189 -> 169),
//  * workgroups begin at different places of K.  All rows of A and W are K
//    apart, so workgroups in step ask the same few channels.  The eight
//    workgroups that begin on the eight XCDs together begin at the same k; the
//    next eight one chunk of 256 bytes later, whose A is then still in L2, or
//    two where rows are 8 or 16 KB apart, so that one chunk does not leave the
//    channel.  With the XCDs spread over K as well rows of a multiple of 16 KB
//    met again: 57344 x 8192, 32 rows 183 -> 165 us; 16384 x 16384, 7 rows 123
//    -> 89; 28672 x 4096, 45 rows 44.1 -> 43.2.  One chunk or two: 28672 x 4096
//    44.0 / 43.2, 8192 x 8192 in 4 parts 27.0 / 24.2, but 16384 x 2048 19.7 /
//    20.4 and, 128 rows of A, whose panel then leaves the L2s, 106496 x 16384
//    808 / 840.  Short parts of rows of 32 KB have too few places for that and
//    stay spread: 4096 x 16384 in 8, 45 rows 26.0, two chunks 28.3.
#include "skinny_rows.h"

namespace {

constexpr int KC = 128;           // k per chunk: 4 loads of 16 rows
constexpr int DEPTH = 2;          // chunks of weights in flight per wave

// NW waves of T * 16 rows of W each share MT * 16 rows of A through LDS, a
// chunk at a time, two buffers, one barrier a chunk.  blockIdx.y: a part of K,
// whose sums go to ws in f32.  GLU: half of the waves hold the gate's rows, the
// others the same rows of the up matrix, and meet in LDS.
template <int MT, int NW, bool GLU, int T>
__global__ __launch_bounds__(64 * NW, 2) void skinny_gemm_kernel(
    const __hip_bfloat16* __restrict__ a,   // [M, K]
    const __hip_bfloat16* __restrict__ w,   // [N, K]
    __hip_bfloat16* __restrict__ c,         // [M, N], GLU: [M, N / 2]
    float* __restrict__ ws,                 // [splits, M, N] if > 1, or C
                                            // in f32 if c is null
    const int M, const int N, const int K, const int splits) {
  constexpr int THREADS = 64 * NW, PITCH = KC + 8;   // + 8: no bank conflicts
  constexpr int PER = THREADS * 8 / KC;     // rows of A that one load covers
  constexpr int PIECES = (MT * 16 + PER - 1) / PER, ROWS = PIECES * PER;
  constexpr int STAGE = 2 * ROWS * PITCH * 2, MEET = GLU ? NW * MT * 1024 : 0;
  __shared__ __align__(16) char lds[STAGE > MEET ? STAGE : MEET];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, g = lane >> 4;
  // columns of this wave; beyond the last it reads the last ones again
  const int half = GLU ? N / 2 : N;
  constexpr int SIDE = GLU ? NW / 2 : NW;
  const int col0 = (blockIdx.x * SIDE + wave % SIDE) * 16 * T;
  const int row = min(col0, half - 16 * T) + (wave / SIDE) * half;
  const int chunks = K / KC;
  const int c0 = chunks * blockIdx.y / splits;
  const int n = chunks * (blockIdx.y + 1) / splits - c0;
  // where a workgroup begins (see above)
  const int octet = blockIdx.x >> 3;
  const bool two = K % 8192 == 0 ? splits > 1 || MT <= 4 || K == 8192
                                 : splits == 1 && K % 4096 == 0;
  const bool spread = K % 8192 == 0 && K > 8192 && splits > 1 && n <= 32;
  const int first = (spread ? octet + (int)(blockIdx.x & 7) * (n >> 3)
                            : two ? octet * 2 : octet) % n;
  // TURN: a load brings 256 bytes of rows g, 4 + g, ... and 4 KB are turned
  constexpr bool TURN = MT <= 6;
  static_assert(T == 1 || TURN, "more rows of a wave come in whole chunks");
  const __hip_bfloat16* wp = w + (size_t)(row + (TURN ? g : r)) * K + c0 * KC +
                             (TURN ? r : g) * 8;
  const size_t hop = TURN ? (size_t)4 * K : 32;
  constexpr int LOADS = T * KC / 32;
  __shared__ __align__(16) __hip_bfloat16 turned[TURN ? NW * T * 16 * PITCH : 8];
  __hip_bfloat16* own = turned + (TURN ? wave * T * 16 * PITCH : 0);
  const __hip_bfloat16* ap[PIECES];
#pragma unroll
  for (int p = 0; p < PIECES; ++p)
    ap[p] = a + (size_t)min((tid / (KC / 8)) + p * PER, M - 1) * K + c0 * KC +
            (tid % (KC / 8)) * 8;
  __hip_bfloat16* buf[2];
  buf[0] = (__hip_bfloat16*)lds;
  buf[1] = buf[0] + ROWS * PITCH;
  const int put = (tid / (KC / 8)) * PITCH + (tid % (KC / 8)) * 8;

  f32x4 acc[T][MT] = {};
  sg_u4 wr[DEPTH][LOADS], ar[PIECES], a0[PIECES];
#define SG_W(s, at)                                                        \
  do {                                                                     \
    const int off = sg_turn(at, first, n) * KC;                            \
    _Pragma("unroll") for (int h = 0; h < LOADS; ++h)                      \
        wr[s][h] = sg_load(wp + off + h * hop);                            \
  } while (0)
#define SG_A(regs, at)                                                     \
  do {                                                                     \
    const int off = sg_turn(at, first, n) * KC;                            \
    _Pragma("unroll") for (int p = 0; p < PIECES; ++p)                     \
        regs[p] = sg_load(ap[p] + off);                                    \
  } while (0)
#define SG_PUT(b, regs)                                                    \
  do {                                                                     \
    _Pragma("unroll") for (int p = 0; p < PIECES; ++p)                     \
        *reinterpret_cast<sg_u4*>((b) + put + p * PER * PITCH) = regs[p];  \
  } while (0)
#define SG_MATH(s, b)                                                      \
  do {                                                                     \
    sg_u4 f[LOADS];                                                        \
    if (TURN) {                                                            \
      _Pragma("unroll") for (int h = 0; h < LOADS; ++h)                    \
          *reinterpret_cast<sg_u4*>(own + (h * 4 + g) * PITCH + r * 8) =   \
              wr[s][h];                                                    \
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");               \
      __builtin_amdgcn_wave_barrier();                                     \
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");               \
    }                                                                      \
    _Pragma("unroll") for (int h = 0; h < LOADS; ++h)                      \
        f[h] = TURN ? sg_load(own + (h / 4 * 16 + r) * PITCH +             \
                              h % 4 * 32 + g * 8)                          \
                    : wr[s][h];                                            \
    _Pragma("unroll") for (int h = 0; h < KC / 32; ++h)                    \
    _Pragma("unroll") for (int i = 0; i < MT; ++i) {                       \
      const sg_u4 x = sg_load((b) + (i * 16 + r) * PITCH + h * 32 + g * 8); \
      _Pragma("unroll") for (int t = 0; t < T; ++t)                        \
          acc[t][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(             \
              sg_frag(x), sg_frag(f[t * (KC / 32) + h]), acc[t][i], 0, 0, 0); \
    }                                                                      \
  } while (0)

  // everything that the first chunks need is asked for before any wait
  SG_A(a0, 0);
  SG_A(ar, min(1, n - 1));
#pragma unroll
  for (int s = 0; s < DEPTH; ++s) SG_W(s, min(s, n - 1));
  __builtin_amdgcn_sched_barrier(0);
  SG_PUT(buf[0], a0);
  int at = 0;
  for (; at + DEPTH < n; at += DEPTH) {
#pragma unroll
    for (int s = 0; s < DEPTH; ++s) {
      __syncthreads();
      SG_PUT(buf[(s + 1) & 1], ar);
      SG_A(ar, min(at + s + 2, n - 1));
      __builtin_amdgcn_sched_barrier(0);
      SG_MATH(s, buf[s & 1]);
      SG_W(s, min(at + s + DEPTH, n - 1));
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int s = 0; s < DEPTH; ++s) {
    if (at + s < n) {
      __syncthreads();
      SG_PUT(buf[(s + 1) & 1], ar);
      if (at + s + 2 < n) SG_A(ar, at + s + 2);
      __builtin_amdgcn_sched_barrier(0);
      SG_MATH(s, buf[s & 1]);
    }
  }
#undef SG_W
#undef SG_A
#undef SG_PUT
#undef SG_MATH

  // lane l, register q: row 4 * g + q of A's tile, column r of 16 of the wave's
  if (GLU) {
    float* meet = (float*)lds;
#pragma unroll
    for (int t = 0; t < T; ++t) {
      __syncthreads();
#pragma unroll
      for (int i = 0; i < MT; ++i)
        *reinterpret_cast<f32x4*>(&meet[(wave * MT + i) * 256 + lane * 4]) =
            acc[t][i];
      __syncthreads();
      for (int e = tid; e < SIDE * MT * 256; e += THREADS) {
        const int i = (e >> 8) % MT, side = (e >> 8) / MT;
        const int m = i * 16 + ((e >> 6) & 3) * 4 + (e & 3);
        const int col = ((blockIdx.x * SIDE + side) * T + t) * 16 +
                        ((e >> 2) & 15);
        if (m < M && col < half)
          c[(size_t)m * half + col] =
              f2bf(silu(meet[e]) * meet[e + SIDE * MT * 256]);
      }
    }
  } else if (col0 < N) {
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int m = i * 16 + g * 4 + q, col = col0 + t * 16 + r;
          if (m >= M) continue;
          if (splits > 1)
            ws[((size_t)blockIdx.y * M + m) * N + col] = acc[t][i][q];
          else if (c)
            c[(size_t)m * N + col] = f2bf(acc[t][i][q]);
          else
            ws[(size_t)m * N + col] = bf2f(f2bf(acc[t][i][q]));
        }
  }
}

__global__ void reduce_splits_kernel(const float* __restrict__ ws,
                                     __hip_bfloat16* __restrict__ c,
                                     const int splits, const long mn) {
  const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= mn) return;
  f32x4 v[1] = {};
  add_parts<8>(v, splits, [&](int s, int) {
    return *reinterpret_cast<const f32x4*>(ws + (size_t)s * mn + i);
  });
  union { __hip_bfloat16 e[4]; uint2 u; } o;
#pragma unroll
  for (int j = 0; j < 4; ++j) o.e[j] = f2bf(v[0][j]);
  *reinterpret_cast<uint2*>(c + i) = o.u;
}

template <int MT, int NW, bool GLU, int T = 1>
void launch_tiles(__hip_bfloat16* c, float* ws, const __hip_bfloat16* a,
                  const __hip_bfloat16* w, int M, int N, int K, int splits,
                  hipStream_t stream) {
  const int cols = NW * T * (GLU ? 8 : 16), out = GLU ? N / 2 : N;
  skinny_gemm_kernel<MT, NW, GLU, T>
      <<<dim3((out + cols - 1) / cols, splits), dim3(64 * NW), 0, stream>>>(
          a, w, c, ws, M, N, K, splits);
}

// Up to 64 rows: 32 rows of W a wave where that makes one round of the chip of
// what would be one and a part.  A CU with two workgroups reads no faster than
// with one, so that the others wait, and A passes L2 half as often (64 rows:
// 51200 x 5120 108 -> 95 us, 45056 x 4096 77 -> 67, 36864 x 4096 75 -> 62; over
// 2048 to 8192 k: to 40960 columns 0.76 to 0.91, to 53248 0.84 to 1.03, 57344
// 0.90 to 1.05; 65536, two whole rounds, 0.92 to 1.07, 69632 1.09 to 1.22).
template <int MT, bool GLU>
void launch_wide(__hip_bfloat16* c, float* ws, const __hip_bfloat16* a,
                 const __hip_bfloat16* w, int M, int N, int K, int splits,
                 hipStream_t stream) {
  if (MT <= 4 && splits == 1 && N > 32768 && N <= 57344 &&
      (GLU ? N / 2 : N) % 32 == 0)
    launch_tiles<MT, 8, GLU, MT <= 4 ? 2 : 1>(c, ws, a, w, M, N, K, splits,
                                             stream);
  else
    launch_tiles<MT, 8, GLU>(c, ws, a, w, M, N, K, splits, stream);
}

}  // namespace

// ---------------------------------------------------------------------------
// C launchers (torch glue lives in gemm_bindings.h)

// c may be null where nothing is split (splits == 1): ws is C then, in f32.
extern "C" void launch_skinny_gemm(void* c, void* ws, const void* a,
                                   const void* w, int M, int N, int K,
                                   int waves, int splits, int glu,
                                   hipStream_t stream) {
  const __hip_bfloat16* ap = (const __hip_bfloat16*)a;
  const __hip_bfloat16* wp = (const __hip_bfloat16*)w;
  __hip_bfloat16* cp = (__hip_bfloat16*)c;
  float* wsp = (float*)ws;
  const int mt = (M + 15) >> 4;
#define SG_GO(MT)                                                          \
  do {                                                                     \
    if (glu)                                                               \
      launch_wide<MT, true>(cp, wsp, ap, wp, M, N, K, 1, stream);          \
    else                                                                   \
      launch_wide<MT, false>(cp, wsp, ap, wp, M, N, K, splits, stream);    \
  } while (0)
#define SG_HALF(MT, GLU)                                                   \
  launch_tiles<MT, 4, GLU>(cp, wsp, ap, wp, M, N, K, GLU ? 1 : splits, stream)
  if (waves == 0) {             // the kernel of a few rows
    if (glu)
      launch_skinny_rows<true>(cp, ap, wp, M, N, K, stream);
    else if ((N <= 2048 && K >= 4096) ||
             (M == 1 && N > 4096 && N <= 6144 && K >= 8192))
      launch_skinny_rows<false, true>(cp, ap, wp, M, N, K, stream,
                                      cp ? nullptr : wsp);
    else
      launch_skinny_rows<false>(cp, ap, wp, M, N, K, stream,
                                cp ? nullptr : wsp);
  } else if (mt <= 1 && waves == 4) {
    if (glu) SG_HALF(1, true);
    else SG_HALF(1, false);
  } else if (mt <= 2 && waves == 4) {
    if (glu) SG_HALF(2, true);
    else SG_HALF(2, false);
  } else if (mt <= 1) SG_GO(1);
  else if (mt <= 2) SG_GO(2);
  else if (mt <= 3 && waves == 4 && glu) SG_HALF(3, true);
  else if (mt <= 4 && waves == 4 && glu) SG_HALF(4, true);
  else if (mt <= 3) SG_GO(3);
  else if (mt <= 4) SG_GO(4);
  else if (mt <= 6) SG_GO(6);
  else if (mt <= 8) SG_GO(8);
  else if (mt <= 12)
    launch_tiles<12, 8, false>(cp, wsp, ap, wp, M, N, K, splits, stream);
  else
    launch_tiles<16, 8, false>(cp, wsp, ap, wp, M, N, K, splits, stream);
#undef SG_GO
#undef SG_HALF
}

extern "C" void launch_reduce_splits(void* c, const void* ws, int splits,
                                     long mn, hipStream_t stream) {
  const int threads = 256;
  const long vecs = mn / 4;     // N is a multiple of 32
  reduce_splits_kernel<<<dim3((vecs + threads - 1) / threads), dim3(threads),
                         0, stream>>>((const float*)ws, (__hip_bfloat16*)c,
                                      splits, mn);
}
