// Paged decode attention (one query token per sequence, GQA) on MFMA.
//
// Cache layout [num_blocks, Hkv, 16, D]: a (page, head) tile is contiguous
// (4 KB of bf16 at D = 128). Reading the pages is all that cannot be avoided;
// the kernel is organised around keeping enough of those reads in flight.
//
// A block takes the query heads of one KV head of one sequence (or of one of
// several splits of its context) and its waves take pairs of pages in turn,
// each wave in LDS of its own: bf16 pages arrive by LDS-direct loads, two
// pairs (32 KB) in flight per wave without a register or a barrier; E4M3 pages
// pass through registers and are widened (exactly) on the way.
//
// The tiles are transposed: S^T = K Q^T on v_mfma_f32_16x16x32_bf16 puts one
// query head per lane column, and the score registers of a page pair are
// already the B operand of O^T += V^T P^T (contraction index 8 g + j: key
// 4 g + j of the first page for j < 4, of the second after that); V is read
// from its row-major tile by the transposing LDS loads. K and q are bf16, so
// their products are exact and the scores fp32; the softmax weights stay 24
// bits wide: they enter as three bf16 parts (high, middle, low) whose products
// are summed in fp32. A group of up to five heads has its three parts side by
// side in the 16 columns of one product (the query is repeated); six to eight
// heads put two parts there and the third through a second product.
//
// Measured (32 query and 8 KV heads of 128; before it a wave per query head
// walked the pages with vector dot products): 256 sequences of 2048 +- 60%
// tokens 739 -> 358 us (6.0 TB/s of pages), all of 2048 609 -> 330 us (6.5);
// 512 of 576 341 -> 198 us; E4M3, 96 of 3000 385 -> 119 us; one of 560 9.4 ->
// 7.6 us, of 7000 45 -> 12 us; 64 / 8 heads, 64 of 600 71 -> 29 us. The page
// loads are non-temporal: a step's pages pass once and a model's do not fit
// the caches (temporal, the first four take 392, 366, 216 and 131 us; only
// pages still cached from the last call, 64 of 1000 alone, gain, 47 / 55).
//
// Splits are merged by paged_attention_reduce_kernel. Numerics oracle:
// ops/torch_ref.paged_attention_decode.
#include "mfma_attention.h"

using namespace mfma_attn;

extern "C" int ks_paged_decode_splits(int num_seqs, int num_kv_heads,
                                      int max_blocks) {
  return decode_splits(num_seqs, num_kv_heads, max_blocks);
}

extern "C" hipError_t ks_paged_attention_decode(
    void* out, const void* q, const void* k_cache, const void* v_cache,
    const void* block_tables, const void* context_lens, float scale,
    int num_seqs, int num_heads, int num_kv_heads, int head_dim,
    int max_blocks, int block_size, long q_row_stride, int n_splits,
    void* part_out, void* part_ml, int window, int fp8, hipStream_t stream) {
  if (block_size != PAGE) return hipErrorInvalidValue;
  const int group = num_heads / num_kv_heads;
  if (group < 1 || group > (fp8 ? 4 : 8)) return hipErrorInvalidValue;
  if (num_seqs == 0) return hipSuccess;
  if (n_splits < 1 || !part_out || !part_ml) n_splits = 1;
  const DecodeArgs p{out, q, k_cache, v_cache,
                     (const int*)block_tables, (const int*)context_lens, scale,
                     num_heads, num_kv_heads, group, max_blocks, q_row_stride,
                     n_splits, (float*)part_out, (float*)part_ml, window,
                     head_dim, head_dim, nullptr, Extra{}};
  const bool aligned = (((uintptr_t)k_cache | (uintptr_t)v_cache) & 15) == 0;
  if (head_dim == 128) {
    if (fp8) return launch_decode<128, PAGES_FP8>(p, num_seqs, stream);
    if (aligned) return launch_decode<128, PAGES_DMA>(p, num_seqs, stream);
    return launch_decode<128, PAGES_REG>(p, num_seqs, stream);
  }
  if (head_dim == 64 && !fp8) {
    if (aligned) return launch_decode<64, PAGES_DMA>(p, num_seqs, stream);
    return launch_decode<64, PAGES_REG>(p, num_seqs, stream);
  }
  return hipErrorInvalidValue;
}
