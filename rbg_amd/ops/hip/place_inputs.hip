// A decode step's inputs, as the host sent them, to where its captured launches
// read them: the sequences' fields, and their page tables in rows of the captured
// width, with page 0 beyond a table and for the rows that pad the batch.  One
// launch in place of two copies and a fill, each of which takes 2 to 4 us.  From the
// host's pinned memory it needs no copy before it, of 4 to 5 us, 6 us behind which it
// began (a step of 128 sequences 1931 -> 1910 us, of 45 1044 -> 1028, of 64 of qwen 32b
// 1193 -> 1177).
#include "host_read.h"

namespace {

// the new ones are in the host's memory
__global__ __launch_bounds__(256) void place_inputs_kernel(
    long* __restrict__ fields, const long* __restrict__ new_fields,
    const int count, int* __restrict__ tables,     // [rows, width]
    const int* __restrict__ new_tables,            // [seqs, used]
    const int rows, const int width, const int seqs, const int used) {
  const int at = blockIdx.x * 256 + threadIdx.x;
  const int row = at / width, col = at % width;
  const bool held = row < seqs && col < used;
  if (at < count) fields[at] = host_read(new_fields + at);
  if (at >= rows * width) return;
  tables[at] = held ? host_read(new_tables + row * used + col) : 0;
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
      (const int*)new_tables, rows, max(width, 1), seqs, used);
}
