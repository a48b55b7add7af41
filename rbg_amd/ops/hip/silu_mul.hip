// Fused SwiGLU activation: out = silu(x[:, :I]) * x[:, I:].
// Pure HBM-bound elementwise op — grid-stride, 16-byte bf16 vectors
// (guide Appendix B elementwise pattern).
#include "common.h"

namespace {

__global__ void silu_mul_kernel(__hip_bfloat16* __restrict__ out,   // [T, I]
                                const __hip_bfloat16* __restrict__ x,  // [T, 2I]
                                const int inter, const long total_vec) {
  const long stride = (long)gridDim.x * 256;
  const int nvec_row = inter / 8;
  for (long i = blockIdx.x * 256l + threadIdx.x; i < total_vec;
       i += stride) {
    const long row = i / nvec_row;
    const int col = (int)(i % nvec_row) * 8;
    Bf16x8U g, u, o;
    g.u = *reinterpret_cast<const uint4*>(x + row * 2 * inter + col);
    u.u = *reinterpret_cast<const uint4*>(x + row * 2 * inter + inter + col);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float gv = bf2f(g.e[j]);
      const float silu = gv / (1.f + __expf(-gv));
      o.e[j] = f2bf(silu * bf2f(u.e[j]));
    }
    *reinterpret_cast<uint4*>(out + row * inter + col) = o.u;
  }
}

// The same of the f32 sums [parts, T, 2I] that a split GEMM left, for decode
// batches: the reduction's launch (2 us) and its result's way through memory
// are saved.
template <int U>
__global__ void silu_parts_kernel(__hip_bfloat16* __restrict__ out,  // [T, I]
                                  const float* __restrict__ x,
                                  const int parts, const int inter,
                                  const long total_vec) {
  const long i = blockIdx.x * 256l + threadIdx.x;
  if (i >= total_vec) return;
  const int nvec_row = inter / 4;
  const long row = i / nvec_row;
  const int col = (int)(i % nvec_row) * 4;
  const float* p = x + row * 2 * inter + col;
  const size_t step = (size_t)total_vec * 8;
  f32x4 v[2] = {};                // gate, up
  add_parts<U>(v, parts, [&](int s, int i) {
    return *reinterpret_cast<const f32x4*>(p + s * step + i * inter);
  });
  union { __hip_bfloat16 e[4]; uint2 u; } o;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    o.e[j] = f2bf(v[0][j] / (1.f + __expf(-v[0][j])) * v[1][j]);
  *reinterpret_cast<uint2*>(out + row * inter + col) = o.u;
}

}  // namespace

extern "C" {

void launch_silu_parts(void* out, const void* x, int parts, int tokens,
                       int inter, hipStream_t stream) {
  const long vecs = (long)tokens * (inter / 4);
  auto go = [&](auto kernel) {
    kernel<<<dim3((vecs + 255) / 256), dim3(256), 0, stream>>>(
        (__hip_bfloat16*)out, (const float*)x, parts, inter, vecs);
  };
  // parts on their way: eight, but two where there are many threads (16 rows of 10240
  // in 6 parts 3.2 / 3.6 us; 200 of 13696 in 2 7.0 / 6.4, 600 of 5120 in 2 7.5 / 6.9)
  if (vecs <= 1 << 17) go(silu_parts_kernel<8>);
  else go(silu_parts_kernel<2>);
}

void launch_silu_mul(void* out, const void* x, int tokens, int inter,
                     hipStream_t stream) {
  const long total_vec = (long)tokens * (inter / 8);
  int blocks = (int)((total_vec + 255) / 256);
  if (blocks > 8192) blocks = 8192;   // grid-stride covers the rest
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(silu_mul_kernel, dim3(blocks), dim3(256), 0, stream,
                     (__hip_bfloat16*)out, (const __hip_bfloat16*)x, inter,
                     total_vec);
}

}  // extern "C"
