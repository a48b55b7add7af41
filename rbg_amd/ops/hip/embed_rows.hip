// Rows of an embedding table in bf16.  Bound by latency for a decode batch (one
// load of the id, one of the row), by memory for a prompt: a workgroup per
// token, 16 bytes a thread.  An id below 0 counts from the end, as an index of a
// tensor does; one outside the table has no row and gives NaN.
#include "common.h"

namespace {

__global__ __launch_bounds__(512) void embed_rows_kernel(
    __hip_bfloat16* __restrict__ out,           // [T, width]
    const __hip_bfloat16* __restrict__ table,   // [rows, width]
    const long* __restrict__ ids, const long rows, const int width) {
  long id = ids[blockIdx.x];
  if (id < 0) id += rows;
  const bool there = id >= 0 && id < rows;
  const uint4* src =
      reinterpret_cast<const uint4*>(table + (there ? id : 0) * width);
  uint4* dst = reinterpret_cast<uint4*>(out + (size_t)blockIdx.x * width);
  const uint4 none = {0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u};
  for (int i = threadIdx.x; i < width / 8; i += 512)
    dst[i] = there ? src[i] : none;
}

}  // namespace

extern "C" void launch_embed_rows(void* out, const void* table,
                                  const void* ids, long rows, int width,
                                  int tokens, hipStream_t stream) {
  const int threads = min(512, (width / 8 + 63) / 64 * 64);
  embed_rows_kernel<<<dim3(tokens), dim3(threads), 0, stream>>>(
      (__hip_bfloat16*)out, (const __hip_bfloat16*)table, (const long*)ids,
      rows, width);
}
