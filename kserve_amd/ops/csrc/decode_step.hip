// The bookkeeping of a decode step beside the model, one launch each: a step
// of few tokens is as long as the launches in it, and these stood for fifteen
// (five copies out of pinned memory, the page-slot arithmetic, the increments).
// Measured with one and 256 rows: 3.4 and 4.2 us (unpack), 4.0 us (advance)
// in place of 15 launches of 4.4 us. The rows may lie in pinned host memory, where
// the kernel reads them itself. The copy ahead of it, and the wait between the two,
// took up to 16 us of a step (us, copied / read in place: 1 row 449.3 / 449.0, 24
// rows 532.8 / 530.6, 96 1031 / 1015, 256 2312 / 2297). Wide tables are bound by the bus
// either way (alone, 96 rows of 4096 pages 47 / 32, 256 of 4096 93 / 80, 2048 of 4096, 33
// MB, 623 / 608), so that no size goes back to the copy.
#include "common.h"
#include "decode_step.h"

namespace {

constexpr int HEAD = 8;  // ints of a staged row before its page table

// Staged rows [rows][stride] ints: token id (64 bits), position (64 bits),
// context length, state slot, page slot, unused, then the page table.
__global__ __launch_bounds__(256) void unpack_decode_rows_kernel(
    const int* __restrict__ staged, const long stride, const int width,
    long* __restrict__ ids, long* __restrict__ positions,
    int* __restrict__ context_lens, int* __restrict__ state_slots,
    int* __restrict__ slots, int* __restrict__ tables, const long table_stride) {
  const int* row = staged + blockIdx.x * stride;
  for (int i = blockIdx.y * 256 + threadIdx.x; i < width; i += gridDim.y * 256)
    tables[blockIdx.x * table_stride + i] = row[HEAD + i];
  if (blockIdx.y == 0 && threadIdx.x == 0) {
    ids[blockIdx.x] = ((long)row[1] << 32) | (unsigned int)row[0];
    positions[blockIdx.x] = ((long)row[3] << 32) | (unsigned int)row[2];
    context_lens[blockIdx.x] = row[4];
    state_slots[blockIdx.x] = row[5];
    slots[blockIdx.x] = row[6];
  }
}

// The next step's inputs: the sampled token (greedy where `random` is null or
// the row's mask is set), the next position with its page slot, the longer
// context and the next seed.
__global__ __launch_bounds__(256) void advance_decode_kernel(
    const long* __restrict__ greedy, const long* __restrict__ random,
    const unsigned char* __restrict__ greedy_mask, long* __restrict__ sampled,
    const NextStep next, long* __restrict__ seeds, const long seed_step, const int rows) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= rows) return;
  const long token = random && !greedy_mask[i] ? random[i] : greedy[i];
  if (sampled) sampled[i] = token;
  const long pos = next.positions[i] + 1;
  write_next(next, i, token, pos, next_slot(next, i, pos));
  if (seeds) seeds[i] += seed_step;
}

}  // namespace

extern "C" hipError_t ks_unpack_decode_rows(const void* staged, long stride, int rows,
                                            int width, void* ids, void* positions,
                                            void* context_lens, void* state_slots,
                                            void* slots, void* tables,
                                            long table_stride, hipStream_t stream) {
  if (rows < 0 || width < 0 || stride < HEAD + width || table_stride < width)
    return hipErrorInvalidValue;
  if (rows == 0) return hipSuccess;
  const int by = width > 2048 ? 8 : (width + 255) / 256;
  hipLaunchKernelGGL(unpack_decode_rows_kernel, dim3(rows, by < 1 ? 1 : by), dim3(256),
                     0, stream, (const int*)staged, stride, width, (long*)ids,
                     (long*)positions, (int*)context_lens, (int*)state_slots,
                     (int*)slots, (int*)tables, table_stride);
  HIP_CHECK_KERNEL();
  return hipSuccess;
}

extern "C" hipError_t ks_advance_decode(const void* greedy, const void* random,
                                        const void* greedy_mask, void* sampled,
                                        void* ids, void* positions,
                                        void* context_lens, void* slots, void* seeds,
                                        long seed_step, const void* tables,
                                        long table_stride, int width, int block,
                                        int rows, hipStream_t stream) {
  if (rows < 0 || width < 1 || block < 1 || (random && !greedy_mask))
    return hipErrorInvalidValue;
  if (rows == 0) return hipSuccess;
  const NextStep next{(long*)ids,         (long*)positions,   (int*)context_lens,
                      (int*)slots,        (const int*)tables, table_stride, width, block};
  hipLaunchKernelGGL(advance_decode_kernel, dim3((rows + 255) / 256), dim3(256), 0,
                     stream, (const long*)greedy, (const long*)random,
                     (const unsigned char*)greedy_mask, (long*)sampled, next, (long*)seeds,
                     seed_step, rows);
  HIP_CHECK_KERNEL();
  return hipSuccess;
}
