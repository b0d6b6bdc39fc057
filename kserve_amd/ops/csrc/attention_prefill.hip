// Flash-style prefill attention (bf16, GQA, varlen) on MFMA: rows of the
// current batch (flash_prefill_varlen) or pages of the KV cache
// (context_prefill_varlen: chunked prefill, prefix reuse, draft verification).
//
// The tiles are transposed: S^T = K Q^T puts one query per lane column of
// v_mfma_f32_32x32x16_bf16, so the running maximum, sum and rescale factor are
// per-lane scalars, and the 16 score registers of a lane are already the B
// operand of O^T += V^T P^T: the contraction runs over keys in the
// accumulator's own order (lane half h, element j -> key 4h + j, then
// 8 + 4h + j of a 16-key chunk), and V is read from its row-major LDS tile in
// that order by the transposing LDS loads (ds_read_b64_tr_b16). The weights
// never leave registers.
//
// A block is 4 waves of 32 queries and shares double-buffered tiles of 64 keys
// that the LDS-direct loads fill while the other buffer is computed on (they run
// under K Q^T and the softmax: the compiler waits for them ahead of the
// transposing reads of V; without that wait it moves those reads up and the tile
// takes 10% longer); the XOR swizzles are on the source side of those loads. With
// several query heads per KV head the waves take up to four heads of one group
// over the same queries (equal causal ranges, and a K/V tile is fetched once for
// the group); otherwise consecutive queries of one head. Few queries behind a long
// context are split over its keys.
//
// What bounds it: per 64 keys and 32 queries a wave issues 32 MFMAs (1024 cycles of
// its matrix core), reads 32 KB of LDS operands (256 cycles of the unit's LDS, for 8
// waves as much as the products of two) and has 32 exponentials and about 130 further
// vector instructions per lane (1050 cycles); two waves per SIMD overlap the three.
// The sign of the scale in the query, the exponent as one multiply-add, a maximum
// that is followed in steps of 2^8, tile addresses from scalars, and keys read six
// products ahead took 700 vector cycles and most waits off a tile. Measured (32 query
// and 8 KV heads of 128, causal; the 16x16x32 kernel with one head per block before,
// then before and with those; waves with products ahead of waves with vector
// instructions take another 1 to 4 % off): 1 x 8191 tokens 2497 / 621 / 557 us (990
// TFLOP/s), 8 x 2048 1280 / 373 / 329 us, 16 x 500 77 / 72 us; 2 x 1000 queries over 13000
// paged keys 2441 / 484 / 438 us (E4M3 pages 2596 / 567 / 500); 8 x 500, 12 heads of 64,
// bidirectional 20 / 17 us, 64 x 123 level at 13; fp32 scores, 4 x 2000, 16 / 4 heads
// 239 / 223 us.
//
// Replaces the vLLM flash prefill the reference delegates to. Numerics oracles:
// ops/torch_ref.flash_prefill_varlen and context_attention_varlen.
#include "mfma_attention.h"

namespace {

using namespace mfma_attn;

// adds the parts of prefill_attention_kernel's keys: 32 lanes per (token, head),
// 4 of 128 columns each. Parts without a tile wrote no sums; the others count even
// where their weights are NaN (by bits: a comparison of a NaN is the compiler's to
// choose here), so that NaNs come out as from one part.
__global__ __launch_bounds__(256) void prefill_attention_merge_kernel(
    short* __restrict__ out, const float* __restrict__ part_out,
    const float* __restrict__ part_ml, const int n_splits, const long rows) {
  constexpr int D = 128;
  const long row = blockIdx.x * 8L + (threadIdx.x >> 5);
  if (row >= rows) return;
  const int d = (threadIdx.x & 31) * 4;
  auto empty = [](float l) {
    return __builtin_bit_cast(int, l) == __builtin_bit_cast(int, NO_KEYS);
  };
  float top = -3.4e38f;
  for (int s = 0; s < n_splits; ++s) {
    const float2_t ml = *reinterpret_cast<const float2_t*>(part_ml + (s * rows + row) * 2);
    if (!empty(ml[1])) top = fmaxf(top, ml[0]);
  }
  float sum = 0.f;
  f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < n_splits; ++s) {
    const float2_t ml = *reinterpret_cast<const float2_t*>(part_ml + (s * rows + row) * 2);
    if (!empty(ml[1])) {
      const float f = __builtin_amdgcn_exp2f(ml[0] - top);
      sum += f * ml[1];
      acc += f * *reinterpret_cast<const f32x4_t*>(part_out + (s * rows + row) * D + d);
    }
  }
  store4(out, row * D + d, acc * (sum > 0.f ? 1.f / sum : 0.f), 0);
}

// query heads that a block takes
int heads_per_block(int group) { return group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1; }

template <int D, int SRC>
hipError_t launch(PrefillArgs p, int num_seqs, int max_q_len, bool causal,
                  hipStream_t stream) {
  p.hpb = heads_per_block(p.Hq / p.Hkv);
  const int qpb = NWAVES * QW / p.hpb;
  const int tiles = (max_q_len + qpb - 1) / qpb;
  if (tiles == 0 || num_seqs == 0) return hipSuccess;
  const dim3 grid(p.Hq / p.hpb, tiles, num_seqs * p.n_splits);
#define GO(CC, WW)                                                             \
  hipLaunchKernelGGL((prefill_attention_kernel<D, SRC, CC, WW>), grid,         \
                     dim3(256), 0, stream, p)
  const bool win = p.window > 0;
  if constexpr (SRC >= PAGES_DMA) {
    if (win) GO(true, true);
    else GO(true, false);
  } else if (causal) {
    if (win) GO(true, true);
    else GO(true, false);
  } else {
    if (win) GO(false, true);
    else GO(false, false);
  }
#undef GO
  HIP_CHECK_KERNEL();
  if (p.n_splits > 1) {
    hipLaunchKernelGGL(prefill_attention_merge_kernel, dim3((unsigned)((p.rows + 7) / 8)),
                       dim3(256), 0, stream, (short*)p.out, p.part_out, p.part_ml,
                       p.n_splits, p.rows);
    HIP_CHECK_KERNEL();
  }
  return hipSuccess;
}

bool aligned16(const void* a, const void* b) {
  return (((uintptr_t)a | (uintptr_t)b) & 15) == 0;
}

}  // namespace

// key parts for such a call (what its workspace is sized for)
extern "C" int ks_context_prefill_splits(int num_seqs, long rows, int max_q_len, int Hq,
                                         int Hkv, int max_nb, int window) {
  if (num_seqs < 1 || max_q_len < 1 || Hkv < 1 || Hq % Hkv != 0) return 1;
  const int hpb = heads_per_block(Hq / Hkv), qpb = NWAVES * QW / hpb;
  const long blocks = (long)(Hq / hpb) * ((max_q_len + qpb - 1) / qpb) * num_seqs;
  long keys = (long)max_nb * PAGE;
  if (window > 0 && keys > (long)window + qpb) keys = (long)window + qpb;
  return prefill_splits(blocks, (int)((keys + KT - 1) / KT), rows);
}

extern "C" hipError_t ks_context_prefill_varlen(
    void* out, const void* q, const void* k_cache, const void* v_cache,
    const void* block_tables, const void* ctx_lens, const void* cu_seqlens_q,
    int num_seqs, int max_q_len, int Hq, int Hkv, int head_dim, int max_nb,
    float scale, long sq, int fp8_cache, int window, long rows, int n_splits,
    void* part_out, void* part_ml, hipStream_t stream) {
  if (head_dim != 128) return hipErrorInvalidValue;
  if (n_splits < 1 || !part_out || !part_ml) n_splits = 1;
  if (Hq % Hkv != 0) return hipErrorInvalidValue;
  PrefillArgs p{out, q, k_cache, v_cache,
                (const int*)cu_seqlens_q, (const int*)ctx_lens,
                (const int*)block_tables, Hq, Hkv, max_nb, 1, score_scale(scale), sq,
                head_dim, head_dim, window, Extra{}, n_splits, rows,
                (float*)part_out, (float*)part_ml};
  if (fp8_cache) return launch<128, PAGES_FP8>(p, num_seqs, max_q_len, true, stream);
  if (aligned16(k_cache, v_cache))
    return launch<128, PAGES_DMA>(p, num_seqs, max_q_len, true, stream);
  return launch<128, PAGES_REG>(p, num_seqs, max_q_len, true, stream);
}

extern "C" hipError_t ks_flash_prefill_varlen(
    void* out, const void* q, const void* k, const void* v,
    const void* cu_seqlens, int num_seqs, int max_seqlen, int Hq, int Hkv,
    int head_dim, float scale, long sq, long sk, long sv, int causal,
    int window, hipStream_t stream) {
  if (head_dim != 128 && head_dim != 64) return hipErrorInvalidValue;
  if (Hq % Hkv != 0) return hipErrorInvalidValue;
  PrefillArgs p{out, q, k, v, (const int*)cu_seqlens,
                nullptr, nullptr, Hq, Hkv, 0, 1, score_scale(scale), sq, sk, sv, window,
                Extra{}, 1, 0, nullptr, nullptr};
  if (sk >= 1L << 26 || sv >= 1L << 26) return hipErrorInvalidValue;
  // LDS-direct loads move 16 aligned bytes per lane
  const bool dma = aligned16(k, v) && sk % 8 == 0 && sv % 8 == 0;
  if (head_dim == 128) {
    if (dma) return launch<128, ROWS_DMA>(p, num_seqs, max_seqlen, causal, stream);
    return launch<128, ROWS_REG>(p, num_seqs, max_seqlen, causal, stream);
  }
  if (dma) return launch<64, ROWS_DMA>(p, num_seqs, max_seqlen, causal, stream);
  return launch<64, ROWS_REG>(p, num_seqs, max_seqlen, causal, stream);
}
