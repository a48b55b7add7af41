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
// rows, hidden], whose own reduction launch this replaces (2 us or more).
// Bound by latency: a row is one workgroup, so it has as many threads as the
// row has 8-byte pieces and every load of a thread is independent; the sums
// stay in registers between the passes (4096 wide, 128 rows: 3.2 us of the
// kernel above, 3.0 of this one, 4.1 from 8 parts).
template <bool PARTS>
__global__ __launch_bounds__(1024) void add_rmsnorm_row_kernel(
    const void* __restrict__ src, __hip_bfloat16* __restrict__ residual,
    const int parts, const int rows, const int hidden, const int threads,
    const __hip_bfloat16* __restrict__ w, __hip_bfloat16* __restrict__ out,
    const float eps) {
  constexpr int MOST = 4;         // pieces of 4 per thread: hidden <= 16384
  const int row = blockIdx.x, tid = threadIdx.x;
  const size_t at = (size_t)row * hidden;
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
      if (PARTS) {
        const float* p = (const float*)src + at + col;
#pragma unroll 8
        for (int s = 0; s < parts; ++s)
          v += *reinterpret_cast<const f32x4*>(p + (size_t)s * rows * hidden);
      } else {
        B4 x;
        x.u = *reinterpret_cast<const uint2*>(
            (const __hip_bfloat16*)src + at + col);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = bf2f(x.e[j]);
      }
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

}  // namespace

extern "C" {

// parts == 0: src is bf16
void launch_add_rmsnorm_rows(void* out, const void* src, void* residual,
                             const void* weight, float eps, int parts,
                             int rows, int hidden, hipStream_t stream) {
  const int threads = min(1024, (hidden / 4 + 63) / 64 * 64);
  auto go = [&](auto kernel) {
    kernel<<<dim3(rows), dim3(threads), 0, stream>>>(
        src, (__hip_bfloat16*)residual, parts, rows, hidden, threads,
        (const __hip_bfloat16*)weight, (__hip_bfloat16*)out, eps);
  };
  if (parts) go(add_rmsnorm_row_kernel<true>);
  else go(add_rmsnorm_row_kernel<false>);
}

void launch_rmsnorm(void* out, void* input, const void* weight, float eps,
                    int tokens, int hidden, hipStream_t stream) {
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
