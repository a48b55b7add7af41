// A decode step's inputs, as the host sent them, to where its captured launches
// read them: the sequences' fields, and their page tables in rows of the captured
// width, with page 0 beyond a table and for the rows that pad the batch.  One
// launch in place of two copies and a fill, each of which takes 2 to 4 us.
#include "common.h"

namespace {

__global__ __launch_bounds__(256) void place_inputs_kernel(
    long* __restrict__ fields, const long* __restrict__ new_fields,
    const int count, int* __restrict__ tables,     // [rows, width]
    const int* __restrict__ new_tables,            // [seqs, used]
    const int rows, const int width, const int seqs, const int used) {
  const int at = blockIdx.x * 256 + threadIdx.x;
  if (at < count) fields[at] = new_fields[at];
  if (at >= rows * width) return;
  const int row = at / width, col = at % width;
  tables[at] = row < seqs && col < used ? new_tables[row * used + col] : 0;
}

}  // namespace

extern "C" void launch_place_inputs(void* fields, const void* new_fields,
                                    int count, void* tables,
                                    const void* new_tables, int rows,
                                    int width, int seqs, int used,
                                    hipStream_t stream) {
  const int most = max(count, rows * width);
  if (most == 0) return;
  place_inputs_kernel<<<dim3((most + 255) / 256), dim3(256), 0, stream>>>(
      (long*)fields, (const long*)new_fields, count, (int*)tables,
      (const int*)new_tables, rows, width, seqs, used);
}
