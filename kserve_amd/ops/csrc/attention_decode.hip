// Paged decode attention (one query token per sequence, GQA) on MFMA.
//
// Cache layout [num_blocks, Hkv, 16, D]: a (page, head) tile is contiguous
// (4 KB of bf16 at D = 128). Reading the pages is all that cannot be avoided;
// the kernel is organised around keeping enough of those reads in flight.
//
// A block takes the query heads of one KV head of one sequence (or of one of
// several splits of its context) and its waves take pairs of pages in turn,
// each wave in LDS of its own, without a barrier: a pair's rows pass through
// registers, and the next pair's loads are under way while one is multiplied.
// E4M3 rows stay bytes in LDS and are widened (exactly) between there and the product:
// half the LDS, so blocks of four waves where contexts are long. LDS-direct loads into a ring of
// two pairs were slower, the more so the shorter the contexts (500 sequences of
// 100, 8 heads: 60 us, 39 here; 24 of 900 29 / 22; 256 of 2048 328 / 332): the
// ring takes twice the LDS, so half the blocks were resident, and the compiler
// waits for all LDS-direct loads before the transposing LDS reads, so it never
// held more than one pair.
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
// Measured (32 query and 8 KV heads of 128, pages not in a cache; before it a
// wave per query head walked the pages with vector dot products): 256 sequences
// of 2048 +- 60% tokens 741 -> 352 us (6.2 TB/s of pages), all of 2048 606 ->
// 332 us (6.5); 512 of 576 341 -> 189 us; E4M3, 96 of 3000 268 -> 93 us, 3000 +-
// 60% 390 -> 108 us (119 as it came to be measured, 112 now); one of 560 12.5 -> 9.7 us, of 7000 66 -> 14.5 us; 64 / 8
// heads, 64 of 600 83 -> 29 us. Short contexts are bound by a block's fixed work
// (about 5 us) and not by the pages: 500 of 100 tokens, 8 heads 98 -> 42 us, E4M3
// 50 -> 31; one or two pages under one query head each are the only ones slower
// than before (1000 of 16, 32 heads 97 -> 83 us where the table is as short, 138
// in a wide one; E4M3 53 -> 72 and 133). The page loads are
// non-temporal: a step's pages pass once and a model's do not fit the caches.
//
// Splits are merged by paged_attention_reduce_kernel. Numerics oracle:
// ops/torch_ref.paged_attention_decode.
#include "mfma_attention.h"

using namespace mfma_attn;

extern "C" int ks_paged_decode_splits(int num_seqs, int num_kv_heads,
                                      int max_blocks, int head_dim, int fp8) {
  return decode_splits(num_seqs, num_kv_heads, max_blocks, fp8 || head_dim <= 64);
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
                     (const int*)block_tables, (const int*)context_lens,
                     score_scale(scale),
                     num_heads, num_kv_heads, group, max_blocks, q_row_stride,
                     n_splits, (float*)part_out, (float*)part_ml, window,
                     head_dim, head_dim, nullptr, Extra{}};
  if (head_dim == 128)
    return fp8 ? launch_decode<128, PAGES_FP8>(p, num_seqs, stream)
               : launch_decode<128, PAGES_REG>(p, num_seqs, stream);
  if (head_dim == 64 && !fp8) return launch_decode<64, PAGES_REG>(p, num_seqs, stream);
  return hipErrorInvalidValue;
}
