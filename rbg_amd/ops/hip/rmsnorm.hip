// RMSNorm kernels (gfx950): y = x * rsqrt(mean(x^2) + eps) * w, with a fused
// residual-add variant.  HBM-bound: bf16 traffic is fully vectorized as
// 16-byte lane accesses (guide Appendix B / Guideline 13); one 256-thread
// block per row, squares accumulated in f32 with a wave+LDS tree.
//
// Capability analog: the RMSNorm the reference delegates to SGLang engines
// (SURVEY §2.3 prefill/decode engine rows).
#include "common.h"

namespace {

template <bool FUSED_ADD>
__global__ void rmsnorm_kernel(__hip_bfloat16* __restrict__ out,      // [T,H]
                               __hip_bfloat16* __restrict__ input,    // [T,H]
                               __hip_bfloat16* __restrict__ residual, // [T,H]
                               const __hip_bfloat16* __restrict__ w,  // [H]
                               const float eps, const int hidden) {
  const int row = blockIdx.x;
  const int tid = threadIdx.x;
  constexpr int nthreads = 256;
  __shared__ float red[nthreads / 64];
  __shared__ float s_inv;

  __hip_bfloat16* in_row = input + (size_t)row * hidden;
  __hip_bfloat16* res_row =
      FUSED_ADD ? residual + (size_t)row * hidden : nullptr;
  __hip_bfloat16* out_row = out + (size_t)row * hidden;

  const int nvec = hidden / 8;   // hidden % 8 == 0 enforced host-side
  float ss = 0.f;
  for (int i = tid; i < nvec; i += nthreads) {
    Bf16x8U xv;
    xv.u = *reinterpret_cast<const uint4*>(in_row + i * 8);
    if (FUSED_ADD) {
      Bf16x8U rv;
      rv.u = *reinterpret_cast<const uint4*>(res_row + i * 8);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float s = bf2f(xv.e[j]) + bf2f(rv.e[j]);
        xv.e[j] = f2bf(s);
        ss += s * s;
      }
      // residual accumulates the sum (pre-norm residual stream)
      *reinterpret_cast<uint4*>(res_row + i * 8) = xv.u;
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float s = bf2f(xv.e[j]);
        ss += s * s;
      }
    }
  }
  // block reduce
  const int lane = tid & 63, wave = tid >> 6;
  ss = wave_sum(ss);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  if (tid == 0) {
    float total = 0.f;
    for (int wv = 0; wv < (nthreads >> 6); ++wv) total += red[wv];
    s_inv = rsqrtf(total / hidden + eps);
  }
  __syncthreads();
  const float inv = s_inv;

  const __hip_bfloat16* src = FUSED_ADD ? res_row : in_row;
  for (int i = tid; i < nvec; i += nthreads) {
    Bf16x8U xv, wv, ov;
    xv.u = *reinterpret_cast<const uint4*>(src + i * 8);
    wv.u = *reinterpret_cast<const uint4*>(w + i * 8);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      ov.e[j] = f2bf(bf2f(xv.e[j]) * inv * bf2f(wv.e[j]));
    *reinterpret_cast<uint4*>(out_row + i * 8) = ov.u;
  }
}

// residual += src; returns its RMS norm: for decode batches.  src is a row of
// bf16, or (PARTS) the f32 sums that the parts of a split GEMM left, [parts,
// rows, hidden], whose own reduction launch this replaces (2 us or more), or
// (ALONE) there is none, and the residual stays as it is.
// Bound by latency: a row is one workgroup, so it has as many threads as the
// row has 8-byte pieces, to 1024; every load of a thread, the weight's as well, is
// on its way before the first is used, and the sums stay in registers between the
// passes (4096 wide: 8 rows 2.5 us alone, 3.4 from 8 parts, where loads after the
// barrier and pieces in turn took 2.9 and 3.8; 128 rows 2.6, 5.3, before 3.0, 5.7).
enum NormSource { NORM_ALONE, NORM_ROWS, NORM_PARTS };

template <int SOURCE, int MOST, int U>
__global__ __launch_bounds__(1024) void add_rmsnorm_row_kernel(
    const void* __restrict__ src, __hip_bfloat16* __restrict__ residual,
    const int parts, const int rows, const int hidden, const int threads,
    const __hip_bfloat16* __restrict__ w, __hip_bfloat16* __restrict__ out,
    const float eps) {
  const int row = blockIdx.x, tid = threadIdx.x, waves = threads >> 6;
  const size_t at = (size_t)row * hidden;
  __shared__ __align__(16) float red[16];
  union B4 { uint2 u; __hip_bfloat16 e[4]; };
  B4 x[MOST], r[MOST], g[MOST], sum[MOST];
  f32x4 v[MOST] = {};
  int col[MOST];                  // beyond the row: its end again, to no use
#pragma unroll
  for (int i = 0; i < MOST; ++i) {
    col[i] = min((i * threads + tid) * 4, hidden - 4);
    r[i].u = *reinterpret_cast<const uint2*>(residual + at + col[i]);
    if (SOURCE == NORM_ROWS)
      x[i].u = *reinterpret_cast<const uint2*>(
          (const __hip_bfloat16*)src + at + col[i]);
    g[i].u = *reinterpret_cast<const uint2*>(w + col[i]);
  }
  if (tid < 16 && tid >= waves) red[tid] = 0.f;
  if (SOURCE == NORM_PARTS)
    add_parts<U>(v, parts, [&](int s, int i) {
      return *reinterpret_cast<const f32x4*>(
          (const float*)src + at + col[i] + (size_t)s * rows * hidden);
    });
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < MOST; ++i) {
    const bool live = i * threads + tid < hidden >> 2;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float t = (SOURCE == NORM_ROWS ? bf2f(x[i].e[j]) : v[i][j]) +
                      bf2f(r[i].e[j]);
      sum[i].e[j] = f2bf(t);
      ss += live ? t * t : 0.f;
    }
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int k = 0; k < 16; k += 4) {
    const f32x4 t = *reinterpret_cast<const f32x4*>(red + k);
#pragma unroll
    for (int j = 0; j < 4; ++j) total += t[j];
  }
  const float inv = rsqrtf(total / hidden + eps);
#pragma unroll
  for (int i = 0; i < MOST; ++i) {
    if (i * threads + tid < hidden >> 2) {
      B4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        o.e[j] = f2bf(bf2f(sum[i].e[j]) * inv * bf2f(g[i].e[j]));
      *reinterpret_cast<uint2*>(out + at + col[i]) = o.u;
      if (SOURCE != NORM_ALONE)
        *reinterpret_cast<uint2*>(residual + at + col[i]) = sum[i].u;
    }
  }
}

// The same of parts for many long rows, which fill the chip only while two workgroups
// of 1024 threads have room on a CU: a piece of the row after another, its residual
// written before the next, the weight read when all are there.  (us, above / this: 300
// rows of 5120 in 4 parts 9.1 / 9.8, of 8192 in 4 13.7 / 12.8, of 12288 in 3 18.2 /
// 15.6, of 16384 in 4 27.2 / 23.6; 600 of 10240 in 2 19.8 / 19.5, of 8192 in 4 22.4 /
// 24.8; 2048 of 10240 in 2 54.9 / 52.3; 256 of 13696 in 6 20.5 / 22.6.)
__global__ __launch_bounds__(1024, 8) void add_rmsnorm_pieces_kernel(
    const float* __restrict__ src, __hip_bfloat16* __restrict__ residual,
    const int parts, const int rows, const int hidden, const int threads,
    const __hip_bfloat16* __restrict__ w, __hip_bfloat16* __restrict__ out,
    const float eps) {
  constexpr int MOST = 4;
  const int tid = threadIdx.x;
  const size_t at = (size_t)blockIdx.x * hidden;
  __shared__ float red[16];
  union B4 { uint2 u; __hip_bfloat16 e[4]; };
  B4 sum[MOST];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < MOST; ++i) {
    const int col = (i * threads + tid) * 4;
    if (col < hidden) {
      B4 r;
      r.u = *reinterpret_cast<const uint2*>(residual + at + col);
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
      for (int s = 0; s < parts; ++s)
        v += *reinterpret_cast<const f32x4*>(src + at + col +
                                             (size_t)s * rows * hidden);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float t = v[j] + bf2f(r.e[j]);
        sum[i].e[j] = f2bf(t);
        ss += t * t;
      }
      *reinterpret_cast<uint2*>(residual + at + col) = sum[i].u;
    }
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  float total = 0.f;
  for (int k = 0; k < threads >> 6; ++k) total += red[k];
  const float inv = rsqrtf(total / hidden + eps);
#pragma unroll
  for (int i = 0; i < MOST; ++i) {
    const int col = (i * threads + tid) * 4;
    if (col < hidden) {
      B4 g, o;
      g.u = *reinterpret_cast<const uint2*>(w + col);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        o.e[j] = f2bf(bf2f(sum[i].e[j]) * inv * bf2f(g.e[j]));
      *reinterpret_cast<uint2*>(out + at + col) = o.u;
    }
  }
}

template <int SOURCE>
void norm_rows(void* out, const void* src, void* residual, const void* weight,
               float eps, int parts, int rows, int hidden, hipStream_t stream) {
  auto go = [&](auto kernel, int most) {
    const int threads = (hidden / 4 + 64 * most - 1) / (64 * most) * 64;
    kernel<<<dim3(rows), dim3(threads), 0, stream>>>(
        src, (__hip_bfloat16*)residual, parts, rows, hidden, threads,
        (const __hip_bfloat16*)weight, (__hip_bfloat16*)out, eps);
  };
  constexpr bool PARTS = SOURCE == NORM_PARTS;
  if (PARTS && rows > 256 && hidden > 4096 && (hidden > 8192 || rows <= 512)) {
    const int threads = std::min(1024, (hidden / 4 + 63) / 64 * 64);
    add_rmsnorm_pieces_kernel<<<dim3(rows), dim3(threads), 0, stream>>>(
        (const float*)src, (__hip_bfloat16*)residual, parts, rows, hidden,
        threads, (const __hip_bfloat16*)weight, (__hip_bfloat16*)out, eps);
    return;
  }
  // a few loads on their way are enough, or better, where a second round of workgroups
  // has only some (300 rows of 4096 in 6 parts 10.1 -> 9.2 us; 600 in 4 12.0 -> 13.4)
  if (hidden <= 4096 && rows > 256 && rows <= 512)
    go(add_rmsnorm_row_kernel<SOURCE, 1, 1>, 1);
  else if (hidden <= 4096)
    go(add_rmsnorm_row_kernel<SOURCE, 1, PARTS ? 8 : 1>, 1);
  else if (hidden <= 8192 && PARTS && rows > 512)
    go(add_rmsnorm_row_kernel<SOURCE, 2, PARTS ? 2 : 1>, 2);
  else if (hidden <= 8192)
    go(add_rmsnorm_row_kernel<SOURCE, 2, PARTS ? 8 : 1>, 2);
  else if (hidden <= 12288)
    go(add_rmsnorm_row_kernel<SOURCE, 3, PARTS ? 6 : 1>, 3);
  else
    go(add_rmsnorm_row_kernel<SOURCE, 4, PARTS ? 2 : 1>, 4);
}

}  // namespace

extern "C" {

// parts == 0: src is bf16
void launch_add_rmsnorm_rows(void* out, const void* src, void* residual,
                             const void* weight, float eps, int parts,
                             int rows, int hidden, hipStream_t stream) {
  if (parts)
    norm_rows<NORM_PARTS>(out, src, residual, weight, eps, parts, rows, hidden,
                          stream);
  else
    norm_rows<NORM_ROWS>(out, src, residual, weight, eps, 0, rows, hidden,
                         stream);
}

void launch_rmsnorm(void* out, void* input, const void* weight, float eps,
                    int tokens, int hidden, hipStream_t stream) {
  if (tokens <= 256 && hidden >= 256 && hidden <= 16384) {
    norm_rows<NORM_ALONE>(out, nullptr, input, weight, eps, 0, tokens, hidden,
                          stream);
    return;
  }
  dim3 grid(tokens), block(256);
  hipLaunchKernelGGL(rmsnorm_kernel<false>, grid, block, 0, stream,
                     (__hip_bfloat16*)out, (__hip_bfloat16*)input,
                     (__hip_bfloat16*)nullptr, (const __hip_bfloat16*)weight,
                     eps, hidden);
}

// input := rmsnorm(input + residual); residual := input + residual
void launch_fused_add_rmsnorm(void* input, void* residual, const void* weight,
                              float eps, int tokens, int hidden,
                              hipStream_t stream) {
  dim3 grid(tokens), block(256);
  hipLaunchKernelGGL(rmsnorm_kernel<true>, grid, block, 0, stream,
                     (__hip_bfloat16*)input, (__hip_bfloat16*)input,
                     (__hip_bfloat16*)residual, (const __hip_bfloat16*)weight,
                     eps, hidden);
}

}  // extern "C"
