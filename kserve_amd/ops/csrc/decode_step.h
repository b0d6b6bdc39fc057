// What a decode step leaves for the next one, shared by the kernel that writes it
// and the one that finds the greedy token.
#pragma once

struct NextStep {
  long* ids;  // null: nothing is written
  long* positions;
  int* context_lens;
  int* slots;
  const int* tables;
  long table_stride;
  int width, block;
};

// page slot of a row's token at position `pos`
__device__ __forceinline__ int next_slot(const NextStep& to, long row, long pos) {
  // past the table's end (after a window's last step) the slot is not used
  const long page = min(max(pos / to.block, 0L), (long)to.width - 1);
  return to.tables[row * to.table_stride + page] * to.block + (int)(pos % to.block);
}

__device__ __forceinline__ void write_next(const NextStep& to, long row, long token,
                                           long pos, int slot) {
  to.ids[row] = token;
  to.positions[row] = pos;
  to.context_lens[row] += 1;
  to.slots[row] = slot;
}
