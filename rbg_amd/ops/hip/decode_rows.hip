// Decode layers of a few rows: a norm, a GEMM and what follows in one launch
// (skinny_rows.h).
#include "skinny_rows.h"

// end: 0 plain, 1 GLU, 2 ROPE
extern "C" void launch_norm_rows(
    void* c, const void* src, const void* residual, void* residual_out,
    const void* norm_weight, float eps, const void* w, int M, int N, int K,
    int end, const void* cos_sin, const void* positions, const void* slots,
    void* keys, void* values, int heads, int kv_heads, int page_size,
    hipStream_t stream) {
  const RowsNorm norm{(const __hip_bfloat16*)residual,
                      (const __hip_bfloat16*)norm_weight,
                      (__hip_bfloat16*)residual_out, eps};
  const RowsRope rope{(const float*)cos_sin, (const int*)positions,
                      (const int*)slots,     (__hip_bfloat16*)keys,
                      (__hip_bfloat16*)values, heads, kv_heads, page_size};
#define DR_GO(END)                                                         \
  launch_skinny_rows<END, true>((__hip_bfloat16*)c,                        \
                                (const __hip_bfloat16*)src,                \
                                (const __hip_bfloat16*)w, M, N, K, norm,   \
                                rope, stream)
  if (end == 0) DR_GO(ROWS_PLAIN);
  else if (end == 1) DR_GO(ROWS_GLU);
  else DR_GO(ROWS_ROPE);
#undef DR_GO
}
