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
// tokens 733 -> 389 us (5.6 TB/s of pages), all of 2048 606 -> 365 us (5.9);
// 512 of 576 344 -> 217 us; 64 of 1000 71 -> 48 us; 24 of 900 35 -> 27 us; one
// of 560 9.2 -> 7.4 us, of 7000 45 -> 12 us; E4M3, 96 of 3000 377 -> 128 us;
// 64 / 8 heads, 64 of 600 71 -> 29 us.
//
// Splits are merged by paged_attention_reduce_kernel. Numerics oracle:
// ops/torch_ref.paged_attention_decode.
#include "common.h"
#include "mfma_layouts.h"

namespace {

typedef short s16x4_t __attribute__((ext_vector_type(4)));

constexpr int PAGE = 16;
constexpr float MASKED = -3e38f;
constexpr float NO_MAX = -1e30f;  // above MASKED: an all-masked pair adds 0

// how pages get into LDS
enum Src {
  PAGES_DMA,  // bf16, 16-byte aligned: LDS-direct loads
  PAGES_REG,  // bf16 at any alignment: through registers
  PAGES_FP8,  // E4M3, widened to bf16
};

// 16-byte chunk that chunk c of row r of a tile sits at. K fragments: 16 rows
// at one chunk must hit different banks; V fragments: 4 rows of 32 bytes each.
template <int D>
__device__ __forceinline__ int k_swz(int r) {
  return D == 128 ? (r & 15) : ((r >> 1) & 7);
}
template <int D>
__device__ __forceinline__ int v_swz(int r) {
  return D == 128 ? (r & 7) << 1 : ((r >> 1) & 3) << 1;
}

// over the four lanes that share a column (lane & 15)
__device__ __forceinline__ float column_max(float x) {
  const unsigned int u = __float_as_uint(x);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const unsigned int v = __float_as_uint(
      fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1])));
  const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float column_sum(float x) {
  x += __shfl_xor(x, 16, 64);
  return x + __shfl_xor(x, 32, 64);
}

// the pages of a sequence that are read, in pairs, and how they are split
struct Range {
  int first, last;  // page numbers
  int pairs;
  int splits;       // of the launched ones, those with work
  int per;          // pairs per split
};
__device__ __forceinline__ Range page_range(int ctx, int window, int n_splits,
                                            int waves) {
  Range r;
  const int lo = window > 0 ? max(0, ctx - window) : 0;
  r.first = lo / PAGE;
  r.last = (ctx - 1) / PAGE;
  r.pairs = ctx > 0 ? (r.last - r.first) / 2 + 1 : 0;
  // a pair per wave at least
  r.splits = max(1, min(n_splits, (r.pairs + waves - 1) / waves));
  r.per = (r.pairs + r.splits - 1) / r.splits;
  return r;
}

struct DecodeArgs {
  short* out;               // [S, H, D]
  const short* q;           // [S, H, D], row stride sq
  const void* k_cache;      // [NB, Hkv, 16, D]
  const void* v_cache;
  const int* block_tables;  // [S, max_blocks]
  const int* ctx_lens;      // [S]
  float scale;
  int H, Hkv, group, max_blocks;
  long sq;
  int n_splits;
  float* part_out;  // [S, H, n_splits, D]
  float* part_ml;   // [S, H, n_splits, 2]
  int window;
};

template <int D, int NW, int SRC, bool WIDE>  // WIDE: groups of 6 to 8
__global__ __launch_bounds__(NW * 64) void paged_attention_kernel(
    const DecodeArgs p) {
  constexpr int KC = D / 32;           // contraction chunks of K Q^T
  constexpr int DB = D / 16;           // 16-column blocks of the output
  constexpr int ROWS = 2 * PAGE;       // rows of a stage (a pair of pages)
  constexpr int STAGE = 2 * ROWS * D;  // K rows, then V rows
  constexpr int RING = SRC == PAGES_DMA ? 2 : 1;
  // elements per lane and load, loads per stage and tensor
  constexpr int EPL = SRC == PAGES_FP8 ? 16 : 8;
  constexpr int LPR = D / EPL;  // lanes per row
  constexpr int RPI = 64 / LPR;
  constexpr int NI = ROWS / RPI;

  const int kvh = blockIdx.x, s = blockIdx.y, split = blockIdx.z;
  const int ctx = p.ctx_lens[s];
  const Range rg = page_range(ctx, p.window, p.n_splits, NW);
  if (split >= rg.splits) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, g = lane >> 4;
  const int G = p.group;
  constexpr int PARTS = WIDE ? 2 : 3;
  const int part = col / G;  // of the weights: high, middle, low
  const bool used = part < PARTS;

  __shared__ __attribute__((aligned(16))) short lds[NW][RING][STAGE];
  static_assert(RING * STAGE * 2 >= 8 * (D + 4) * 4 + 64, "merge area");

  bf16x8_t qf[KC];
  {
    const short* qp = p.q + (long)s * p.sq + (long)(kvh * G + col % G) * D + g * 8;
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      short8_t x = *reinterpret_cast<const short8_t*>(qp + c * 32);
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = used ? x[j] : 0;
      qf[c] = __builtin_bit_cast(bf16x8_t, x);
    }
  }

  const int* bt = p.block_tables + (long)s * p.max_blocks;
  const int lrow = lane / LPR, lchunk = lane % LPR;
  struct Pages {
    int a, b;
  };
  // page ids of pair n (past the end: the last page again, as its rows are)
  auto pages_of = [&](int n) {
    const int a = min(rg.first + 2 * n, rg.last), b = min(a + 1, rg.last);
    return Pages{bt[a], bt[b]};
  };
  // where this lane's bytes of load i come from; rows past the context repeat
  // its last one (their weights are 0, their values finite)
  auto src = [&](const void* cache, int n, Pages pg, int i, int chunk) {
    constexpr int ES = SRC == PAGES_FP8 ? 1 : 2;
    const bool second = i >= NI / 2;
    const int number = min(rg.first + 2 * n + (second ? 1 : 0), rg.last);
    const int row = min((i % (NI / 2)) * RPI + lrow, ctx - 1 - number * PAGE);
    return reinterpret_cast<const char*>(cache) +
           ((long)(second ? pg.b : pg.a) * p.Hkv + kvh) * (PAGE * D * ES) +
           (row * D + chunk * EPL) * ES;
  };
  auto load_dma = [&](int n, Pages pg, int slot) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int r = i * RPI + lrow;
      short* dst = &lds[wave][slot][i * RPI * D];
      __builtin_amdgcn_global_load_lds(
          reinterpret_cast<const unsigned int*>(
              src(p.k_cache, n, pg, i, lchunk ^ k_swz<D>(r))),
          reinterpret_cast<unsigned int*>(dst), 16, 0, 0);
      __builtin_amdgcn_global_load_lds(
          reinterpret_cast<const unsigned int*>(
              src(p.v_cache, n, pg, i, lchunk ^ v_swz<D>(r))),
          reinterpret_cast<unsigned int*>(dst + ROWS * D), 16, 0, 0);
    }
  };
  uint4 raw[SRC == PAGES_DMA ? 1 : 2 * NI];
  auto load_reg = [&](int n, Pages pg) {
    if constexpr (SRC != PAGES_DMA) {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        raw[2 * i] = *reinterpret_cast<const uint4*>(src(p.k_cache, n, pg, i, lchunk));
        raw[2 * i + 1] =
            *reinterpret_cast<const uint4*>(src(p.v_cache, n, pg, i, lchunk));
      }
    }
  };
  auto commit = [&]() {
    if constexpr (SRC != PAGES_DMA) {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int r = i * RPI + lrow;
#pragma unroll
        for (int kv = 0; kv < 2; ++kv) {
          short* row = &lds[wave][0][kv * ROWS * D + r * D];
          const int sw = kv ? v_swz<D>(r) : k_swz<D>(r);
          const uint4 x = raw[2 * i + kv];
          if constexpr (SRC == PAGES_REG) {
            *reinterpret_cast<uint4*>(row + (lchunk ^ sw) * 8) = x;
          } else {
            const unsigned int w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              uint4 o;
              o.x = __builtin_bit_cast(unsigned int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[2 * h], 1.0f, false));
              o.y = __builtin_bit_cast(unsigned int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[2 * h], 1.0f, true));
              o.z = __builtin_bit_cast(unsigned int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[2 * h + 1], 1.0f, false));
              o.w = __builtin_bit_cast(unsigned int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[2 * h + 1], 1.0f, true));
              *reinterpret_cast<uint4*>(row + ((2 * lchunk + h) ^ sw) * 8) = o;
            }
          }
        }
      }
    }
  };

  // operand addresses inside a stage (elements)
  int kaddr[KC];
#pragma unroll
  for (int c = 0; c < KC; ++c)
    kaddr[c] = col * D + ((4 * c + g) ^ k_swz<D>(col)) * 8;
  // transposing load: lane i of 16 brings key i/4, columns 4 (i%4) .. + 3 and
  // receives column i of its four keys
  const int vrow = g * 4 + (col >> 2);
  int vaddr[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b)
    vaddr[b] = ROWS * D + vrow * D +
               ((2 * b + ((col & 3) >> 1)) ^ v_swz<D>(vrow)) * 8 + (col & 1) * 4;

  float c2 = p.scale * 1.44269504088896340736f;
  const bool flip = c2 < 0.f;
  c2 = fabsf(c2);
  const int key_lo = p.window > 0 ? ctx - p.window : 0;  // first visible key
  float m = NO_MAX, l = 0.f;
  f32x4_t o[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b) o[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  auto compute = [&](int n, const short* st) {
    f32x4_t sc[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      sc[h] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < KC; ++c)
        sc[h] = mfma16x16x32(
            *reinterpret_cast<const bf16x8_t*>(st + h * PAGE * D + kaddr[c]), qf[c],
            sc[h]);
    }
    if (flip) {
      sc[0] = -sc[0];
      sc[1] = -sc[1];
    }
    const int key0 = (rg.first + 2 * n) * PAGE;
    if (key0 + ROWS > ctx || key0 < key_lo) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = key0 + h * PAGE + g * 4 + r;
          sc[h][r] = key < ctx && key >= key_lo ? sc[h][r] : MASKED;
        }
    }
    float mx = fmaxf(fmaxf(fmaxf(sc[0][0], sc[0][1]), fmaxf(sc[0][2], sc[0][3])),
                     fmaxf(fmaxf(sc[1][0], sc[1][1]), fmaxf(sc[1][2], sc[1][3])));
    mx = column_max(mx);
    if (__any(mx > m)) {
      const float mn = fmaxf(m, mx);
      const float f = __builtin_amdgcn_exp2f((m - mn) * c2);
      m = mn;
      l *= f;
#pragma unroll
      for (int b = 0; b < DB; ++b) o[b] *= f;
    }
    const float mc = m * c2;
    bf16x8_t pf, pl;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float w = __builtin_amdgcn_exp2f(sc[h][r] * c2 - mc);
        l += w;
        // 8 + 8 + 8 bits: hi, mid and lo sum to w exactly
        const __bf16 hi = (__bf16)w;
        const float r1 = w - (float)hi;
        const __bf16 mid = (__bf16)r1;
        const __bf16 lo = (__bf16)(r1 - (float)mid);
        if constexpr (WIDE) {
          pf[h * 4 + r] = part == 0 ? hi : mid;
          pl[h * 4 + r] = part == 0 ? lo : (__bf16)0.f;
        } else {
          pf[h * 4 + r] = part == 0 ? hi : part == 1 ? mid : lo;
        }
      }
#pragma unroll
    for (int b = 0; b < DB; ++b) {
      typedef __attribute__((address_space(3))) s16x4_t lds4_t;
      const short* a0 = st + vaddr[b];
      union {
        s16x4_t h[2];
        bf16x8_t v;
      } a;
      a.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4_t*)a0);
      a.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4_t*)(a0 + PAGE * D));
      o[b] = mfma16x16x32(a.v, pf, o[b]);
      if constexpr (WIDE) o[b] = mfma16x16x32(a.v, pl, o[b]);
    }
  };

  const int n_lo = split * rg.per + wave;
  const int n_hi = min((split + 1) * rg.per, rg.pairs);
  if constexpr (SRC == PAGES_DMA) {
    // s_waitcnt immediates (vmcnt in bits 3:0 and 15:14; no wait on the rest)
    constexpr int NL = 2 * NI;  // loads of one stage
    constexpr int WAIT_STAGE = (0xF << 8) | (0x7 << 4) | (NL & 0xF) | ((NL >> 4) << 14);
    constexpr int WAIT_ALL = (0xF << 8) | (0x7 << 4);
    if (n_lo < n_hi) load_dma(n_lo, pages_of(n_lo), 0);
    if (n_lo + NW < n_hi) load_dma(n_lo + NW, pages_of(n_lo + NW), 1);
    int slot = 0;
    for (int n = n_lo; n < n_hi; n += NW, slot ^= 1) {
      const int next = n + 2 * NW;
      Pages pg{0, 0};
      if (next < n_hi) pg = pages_of(next);
      if (n + NW < n_hi) __builtin_amdgcn_s_waitcnt(WAIT_STAGE);
      else __builtin_amdgcn_s_waitcnt(WAIT_ALL);
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("" ::: "memory");
      compute(n, lds[wave][slot]);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      if (next < n_hi) load_dma(next, pg, slot);
    }
  } else {
    if (n_lo < n_hi) load_reg(n_lo, pages_of(n_lo));
    for (int n = n_lo; n < n_hi; n += NW) {
      commit();
      if (n + NW < n_hi) load_reg(n + NW, pages_of(n + NW));
      compute(n, lds[wave][0]);
    }
  }

  // ---- merge: the parts of the weights, then the waves ----
  l = column_sum(l);
  float* mo = reinterpret_cast<float*>(lds[wave]);  // [8][D + 4], then m and l
  float* mm = mo + 8 * (D + 4);
#pragma unroll
  for (int b = 0; b < DB; ++b) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float x = o[b][r] + __shfl(o[b][r], lane + G, 64);
      if constexpr (!WIDE) x += __shfl(o[b][r], lane + 2 * G, 64);
      o[b][r] = x;
    }
    if (col < G)
      *reinterpret_cast<f32x4_t*>(mo + col * (D + 4) + b * 16 + g * 4) = o[b];
  }
  if (lane < G) {
    mm[lane] = m;
    mm[8 + lane] = l;
  }
  __syncthreads();
  constexpr int WF = RING * STAGE / 2;  // floats between the waves' areas
  const float* all = reinterpret_cast<const float*>(lds);
  for (int i = threadIdx.x; i < G * (D / 4); i += NW * 64) {
    const int h = i / (D / 4), d = i % (D / 4) * 4;
    float top = NO_MAX;
#pragma unroll
    for (int w = 0; w < NW; ++w) top = fmaxf(top, all[w * WF + 8 * (D + 4) + h]);
    float sum = 0.f;
    f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float* a = all + w * WF;
      const float f = __builtin_amdgcn_exp2f((a[8 * (D + 4) + h] - top) * c2);
      sum += f * a[8 * (D + 4) + 8 + h];
      acc += f * *reinterpret_cast<const f32x4_t*>(a + h * (D + 4) + d);
    }
    const long row = (long)s * p.H + kvh * G + h;
    if (rg.splits == 1) {
      const float inv = sum > 0.f ? 1.f / sum : 0.f;
      short4_t w;
#pragma unroll
      for (int r = 0; r < 4; ++r) w[r] = float_to_bf16_bits(acc[r] * inv);
      *reinterpret_cast<short4_t*>(p.out + row * D + d) = w;
    } else {
      const long at = row * p.n_splits + split;
      *reinterpret_cast<f32x4_t*>(p.part_out + at * D + d) = acc;
      if (d == 0) {
        p.part_ml[at * 2] = top * c2;
        p.part_ml[at * 2 + 1] = sum;
      }
    }
  }
}

// Combine split-context partials: one wave per (seq, head); a lane owns D/64
// columns across all splits. Sequences that one split covers are done.
template <int D, int NW>
__global__ __launch_bounds__(256) void paged_attention_reduce_kernel(
    const DecodeArgs p, long total) {
  constexpr int ACC = D / 64;
  const long sh = blockIdx.x * 4L + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (sh >= total) return;
  const Range rg =
      page_range(p.ctx_lens[sh / p.H], p.window, p.n_splits, NW);
  if (rg.splits == 1) return;
  const float* ml = p.part_ml + sh * p.n_splits * 2;
  float m = NO_MAX * 1e6f;
  for (int sp = lane; sp < rg.splits; sp += 64) m = fmaxf(m, ml[sp * 2]);
  m = wave_reduce_max(m);
  float l = 0.f, acc[ACC];
#pragma unroll
  for (int a = 0; a < ACC; ++a) acc[a] = 0.f;
#pragma unroll 4
  for (int sp = 0; sp < rg.splits; ++sp) {
    const float w = __builtin_amdgcn_exp2f(ml[sp * 2] - m);
    l += w * ml[sp * 2 + 1];
    const float* po = p.part_out + (sh * p.n_splits + sp) * D + lane * ACC;
#pragma unroll
    for (int a = 0; a < ACC; ++a) acc[a] += w * po[a];
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
  for (int a = 0; a < ACC; ++a)
    p.out[sh * D + lane * ACC + a] = float_to_bf16_bits(acc[a] * inv);
}

template <int D, int NW, int SRC>
hipError_t launch(const DecodeArgs& p, int num_seqs, hipStream_t stream) {
  const dim3 grid(p.Hkv, num_seqs, p.n_splits);
  if (3 * p.group <= 16)
    hipLaunchKernelGGL((paged_attention_kernel<D, NW, SRC, false>), grid,
                       dim3(NW * 64), 0, stream, p);
  else
    hipLaunchKernelGGL((paged_attention_kernel<D, NW, SRC, true>), grid,
                       dim3(NW * 64), 0, stream, p);
  HIP_CHECK_KERNEL();
  if (p.n_splits > 1) {
    const long sh = (long)num_seqs * p.H;
    hipLaunchKernelGGL((paged_attention_reduce_kernel<D, NW>),
                       dim3((unsigned)((sh + 3) / 4)), dim3(256), 0, stream, p, sh);
    HIP_CHECK_KERNEL();
  }
  return hipSuccess;
}

// Two waves per block: 64 KB of LDS, two blocks per compute unit, so one
// block's first loads run under the other's last ones. (256 sequences of 819 to
// 3277 tokens: 389 us with 2 waves, 390 with 4, 431 with 1; 64 of 400 to 1600:
// 48.4 / 50.0 / 66.4.)
constexpr int WAVES = 2;

}  // namespace

// Context splits for a launch over num_seqs x num_kv_heads: none from 512
// blocks on, which fill the chip (64 sequences, 8 KV heads: 48.4 us unsplit,
// 51.4 with 2 splits, 50.4 with 4; 96 of 3000, E4M3: 128 / 140 / 129), about
// 640 blocks below that (24 sequences of 900: 30.4 us with 3 splits, 27.4 with
// 4, 29.8 with 6; 8 of 600: 9.3 with 8, 11.9 with 16), and at most 32 (one of
// 7000: 12.0 us with 32, 12.8 with 64, 14.7 with 16). A sequence uses as many
// of them as it has page pairs for every wave.
extern "C" int ks_paged_decode_splits(int num_seqs, int num_kv_heads,
                                      int max_blocks) {
  const long base = (long)num_seqs * num_kv_heads;
  if (base <= 0 || base >= 512) return 1;
  long n = (640 + base - 1) / base;
  const long most = ((long)max_blocks + 2 * WAVES - 1) / (2 * WAVES);
  if (n > most) n = most;
  if (n > 32) n = 32;
  return n < 1 ? 1 : (int)n;
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
  const DecodeArgs p{(short*)out, (const short*)q, k_cache, v_cache,
                     (const int*)block_tables, (const int*)context_lens, scale,
                     num_heads, num_kv_heads, group, max_blocks, q_row_stride,
                     n_splits, (float*)part_out, (float*)part_ml, window};
  const bool aligned = (((uintptr_t)k_cache | (uintptr_t)v_cache) & 15) == 0;
  if (head_dim == 128) {
    if (fp8) return launch<128, WAVES, PAGES_FP8>(p, num_seqs, stream);
    if (aligned) return launch<128, WAVES, PAGES_DMA>(p, num_seqs, stream);
    return launch<128, WAVES, PAGES_REG>(p, num_seqs, stream);
  }
  if (head_dim == 64 && !fp8) {
    if (aligned) return launch<64, WAVES, PAGES_DMA>(p, num_seqs, stream);
    return launch<64, WAVES, PAGES_REG>(p, num_seqs, stream);
  }
  return hipErrorInvalidValue;
}
