// Products of few rows with a weight matrix: out[N][M] = x[N][K] w[M][K]^T for
// N <= 256 tokens (decode batches, short prompts), where reading the weights
// is what bounds them. The kernel here takes up to 64 rows, up to 128 of wide
// weights, gate|up products of any number, and rows or K of 2^22 elements and more;
// the rest goes to the tiles of dense_gemm.hip.
//
// A block takes 64 F features (16 F per wave) and all tokens over a range of
// K, in steps of 64: each step's weight and token rows come by LDS-direct
// loads into one slot of a ring, so up to S - 1 steps are in flight behind the
// one that is multiplied, with one barrier per step. K is split over blocks
// until the chip is full; the splits leave fp32 partial sums that a second
// kernel adds in order (no atomics). With GLU the block's rows are as many
// gate as up features and silu(gate) * up leaves it directly.
//
// Measured (us with the reduction, weights not in cache; the library's in
// parentheses): K 4096, M 14336 GLU at 1 row 40 = 5.9 TB/s (67 with the
// activation kernel), at 24 rows 41; K 4096, M 32000 at 1 row 42 (61); K
// 14336, M 4096 at 1 / 24 rows 23 / 24 (27 / 32). Up to 48 rows the loads bound it
// (non-temporal ones took 5 to 10 % off); above, LDS reads and the
// matrix cores of the few blocks that fit, so M of a few thousand or off a multiple of
// 4 KB a row goes back to the library. The kernel before kept a barrier per step behind
// one load in flight and rounded the splits to bf16.
//
// C = W X^T on v_mfma_f32_16x16x32_bf16: a lane ends with four consecutive
// features of one token. LDS rows are 128 bytes; the 16-byte chunk c of row r
// sits at c ^ ((r >> 1) & 7), so 16 rows at one chunk hit different banks; the
// swizzle is on the source side of the loads.
#include "common.h"
#include "mfma_layouts.h"

namespace {

constexpr int BK = 64;  // K per step
constexpr int NWAVES = 4;
constexpr int NT_AUX = 2;  // cache policy of a non-temporal load

enum Epilogue { BF16_OUT, PARTIAL, GLU, CLAMPED };
// gate and up rows: silu(gate) * up or, CLAMPED, gate sigmoid(alpha gate) (up + 1) of
// gate up to a limit and up within it
constexpr bool has_halves(int epi) { return epi == GLU || epi == CLAMPED; }

struct GemmArgs {
  void* out;       // [N][M] bf16; PARTIAL: [splits][N][M] fp32
  const short* x;  // [N][K], row stride xs
  const short* w;  // [M][K]; with halves [2 M][K], gate rows first
  int M, K, N;
  long xs;
  float alpha, limit;  // CLAMPED
  const short* bias;   // BF16_OUT: [M] or null
};

// s_waitcnt with vmcnt <= n (bits 3:0 and 15:14), lgkmcnt 0, expcnt free
constexpr int wait_imm(int n) { return (0x7 << 4) | (n & 0xF) | ((n >> 4) << 14); }

template <int NT, int F, int S, int EPI>
__global__ __launch_bounds__(256) void skinny_gemm_kernel(const GemmArgs p) {
  constexpr int BN = NT * 16, BM = NWAVES * F * 16;
  constexpr int STAGE = (BN + BM) * BK;        // elements
  constexpr int LOADS = (BN + BM) / 8;         // 1 KB loads of a step
  constexpr int NI = (LOADS + NWAVES - 1) / NWAVES;
  constexpr int REM = LOADS % NWAVES;          // waves < REM (or all) issue NI
  static_assert(S >= 2 && S * STAGE * 2 <= 160 * 1024, "ring");
  __shared__ __attribute__((aligned(16))) short ring[S * STAGE];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, g = lane >> 4;
  const int steps = p.K / BK;
  const int lo = (int)((long)steps * blockIdx.y / gridDim.y);
  const int n = (int)((long)steps * (blockIdx.y + 1) / gridDim.y) - lo;
  // Blocks run through their K range in step, and where a row of W is a multiple of
  // 4 KB they would all read the same few memory channels at a time: each pair of
  // blocks starts a step further on and wraps around (us at 1 / 77 rows: K 4096, M
  // 14336 GLU 46.3 / 53.5 -> 40.1 / 45.6, M 32000 47.8 / 59.7 -> 42.2 / 51.0 = 6.2 TB/s;
  // K 2048, M 16384 15.5 -> 13.2; 8192 x 8192 30.4 -> 23.7; level at K 5120; a step a
  // block, or four, leaves some as they were or slower). Not above 64 rows in many
  // parts: the token rows, then as many as W's, are shared through the L2 by blocks
  // at one step (K 14336, M 4096 at 96 / 128 rows 28.1 / 30.0, 29.3 / 34.5 with it).
  const int rot = NT > 4 && gridDim.y > 3 ? 0 : (int)(blockIdx.x / 2) % n;

  // first feature of the block's W rows (with halves: of gate and up rows)
  const int f0 = blockIdx.x * (has_halves(EPI) ? BM / 2 : BM);
  auto w_row = [&](int r) {  // row of w for row r of the tile, clamped
    if constexpr (has_halves(EPI)) {
      const int f = min(f0 + (r < BM / 2 ? r : r - BM / 2), p.M - 1);
      return r < BM / 2 ? f : p.M + f;
    } else {
      return min(f0 + r, p.M - 1);
    }
  };
  // per load: where this lane's 16 bytes of step 0 come from
  const bool full = REM == 0 || wave < REM;
  const char* src[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int r = (wave + i * NWAVES) * 8 + (lane >> 3);  // row of the stage
    const int c = (lane & 7) ^ ((r >> 1) & 7);
    const short* row = r < BN ? p.x + (long)min(r, p.N - 1) * p.xs
                              : p.w + (long)w_row(r - BN) * p.K;
    src[i] = reinterpret_cast<const char*>(row + (long)(lo + rot) * BK + c * 8);
  }
  int issue_slot = 0, to_end = n - rot;
  auto issue = [&]() {  // the next step's loads
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      if (i < NI - 1 || full) {
        const auto* from = reinterpret_cast<const unsigned int*>(src[i]);
        auto* to = reinterpret_cast<unsigned int*>(
            &ring[issue_slot * STAGE + (wave + i * NWAVES) * 8 * BK]);
        if (wave + i * NWAVES < BN / 8)  // token rows: every block reads them
          __builtin_amdgcn_global_load_lds(from, to, 16, 0, 0);
        else
          // past the caches, which hold what the kernels around write and read (us, with
          // / without: llama steps of 64 sequences 632 / 645, hybrid ones of 56 561 /
          // 574); not above 64 rows in parts, whose sums then come back slower (96 E4M3
          // sequences 1006 / 997, 96 of 500 706 / 698, a prompt of 77 tokens 546 / 541)
          __builtin_amdgcn_global_load_lds(from, to, 16, 0,
                                           NT <= 4 || EPI != PARTIAL ? NT_AUX : 0);
        src[i] += BK * 2;
      }
    }
    issue_slot = issue_slot + 1 == S ? 0 : issue_slot + 1;
    if (--to_end == 0) {
#pragma unroll
      for (int i = 0; i < NI; ++i) src[i] -= (long)n * BK * 2;
    }
  };

  f32x4_t acc[F][NT];
#pragma unroll
  for (int f = 0; f < F; ++f)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[f][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int sw = ((col >> 1) & 7);
  const int xat = col * BK, wat = (BN + wave * F * 16 + col) * BK;
  for (int j = 0; j < S - 1 && j < n; ++j) issue();
  int slot = 0;
  for (int j = 0; j < n; ++j) {
    // step j has landed (this wave's part; the barrier covers the others'),
    // and every LDS read of step j - 1 is done
    if (n - 1 - j >= S - 2) {
      if (full) __builtin_amdgcn_s_waitcnt(wait_imm(NI * (S - 2)));
      else __builtin_amdgcn_s_waitcnt(wait_imm((NI - 1) * (S - 2)));
    } else {
      __builtin_amdgcn_s_waitcnt(wait_imm(0));
    }
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (j + S - 1 < n) issue();
    const short* st = &ring[slot * STAGE];
    slot = slot + 1 == S ? 0 : slot + 1;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int c = ((kk * 4 + g) ^ sw) * 8;
      bf16x8_t a[F];
#pragma unroll
      for (int f = 0; f < F; ++f)
        a[f] = *reinterpret_cast<const bf16x8_t*>(st + wat + f * 16 * BK + c);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const bf16x8_t b =
            *reinterpret_cast<const bf16x8_t*>(st + xat + t * 16 * BK + c);
#pragma unroll
        for (int f = 0; f < F; ++f) acc[f][t] = mfma16x16x32(a[f], b, acc[f][t]);
      }
    }
  }

  if constexpr (has_halves(EPI)) {
    // up waves hand their sums to the gate waves through LDS
    __syncthreads();
    f32x4_t* up = reinterpret_cast<f32x4_t*>(ring);  // [2][F][NT][64]
    if (wave >= 2) {
#pragma unroll
      for (int f = 0; f < F; ++f)
#pragma unroll
        for (int t = 0; t < NT; ++t)
          up[(((wave - 2) * F + f) * NT + t) * 64 + lane] = acc[f][t];
    }
    __syncthreads();
    if (wave >= 2) return;
#pragma unroll
    for (int f = 0; f < F; ++f)
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const f32x4_t u = up[((wave * F + f) * NT + t) * 64 + lane];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if constexpr (EPI == GLU) {
            const float x = acc[f][t][r];
            acc[f][t][r] = x / (1.f + __expf(-x)) * u[r];
          } else {
            const float x = fminf(acc[f][t][r], p.limit);
            const float v = fminf(fmaxf(u[r], -p.limit), p.limit);
            acc[f][t][r] = x / (1.f + __expf(-p.alpha * x)) * (v + 1.f);
          }
        }
      }
  }
#pragma unroll
  for (int f = 0; f < F; ++f) {
    const int feat = f0 + (wave * F + f) * 16 + g * 4;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int tok = t * 16 + col;
      if (tok >= p.N || feat >= p.M) continue;
      if constexpr (EPI == PARTIAL) {
        float* o = reinterpret_cast<float*>(p.out) +
                   ((long)blockIdx.y * p.N + tok) * p.M + feat;
        *reinterpret_cast<f32x4_t*>(o) = acc[f][t];
      } else {
        if constexpr (EPI == BF16_OUT) {
          if (p.bias) {
            const short4_t b = *reinterpret_cast<const short4_t*>(p.bias + feat);
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[f][t][r] += bf16_bits_to_float(b[r]);
          }
        }
        short4_t o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = float_to_bf16_bits(acc[f][t][r]);
        *reinterpret_cast<short4_t*>(reinterpret_cast<short*>(p.out) +
                                     (long)tok * p.M + feat) = o;
      }
    }
  }
}

// partial sums of the splits, added in order, and the bias, as bf16; four per thread
__global__ __launch_bounds__(256) void reduce_splits_kernel(
    short* __restrict__ out, const float* __restrict__ part, const long nm,
    const int splits, const short* __restrict__ bias, const int M) {
  const long i = (blockIdx.x * 256L + threadIdx.x) * 4;
  if (i >= nm) return;
  f32x4_t a = *reinterpret_cast<const f32x4_t*>(part + i);
  for (int s = 1; s < splits; ++s)
    a += *reinterpret_cast<const f32x4_t*>(part + s * nm + i);
  if (bias) {
    const short4_t b = *reinterpret_cast<const short4_t*>(bias + i % M);
#pragma unroll
    for (int r = 0; r < 4; ++r) a[r] += bf16_bits_to_float(b[r]);
  }
  short4_t o;
#pragma unroll
  for (int r = 0; r < 4; ++r) o[r] = float_to_bf16_bits(a[r]);
  *reinterpret_cast<short4_t*>(out + i) = o;
}

// token tiles, feature groups per wave and ring slots: two blocks per compute
// unit up to 64 tokens, one with twice the features above
#define FOR_FEW(N, GO)                  \
  if ((N) <= 16) GO(1, 1, 8)            \
  else if ((N) <= 32) GO(2, 1, 6)       \
  else if ((N) <= 48) GO(3, 1, 5)       \
  else if ((N) <= 64) GO(4, 1, 5)
#define FOR_TILE(N, GO)                 \
  FOR_FEW(N, GO)                        \
  else if ((N) <= 96) GO(6, 2, 5)       \
  else if ((N) <= 128) GO(8, 2, 5)      \
  else if ((N) <= 192) GO(12, 2, 4)     \
  else GO(16, 2, 3)

int feature_tile(int N) { return N <= 64 ? 64 : 128; }

}  // namespace

extern "C" int ks_mid_splits(int, int, int);
extern "C" int ks_mid_takes(int, int, int);
extern "C" hipError_t ks_mid_gemm(void*, const void*, const void*, const void*, int, int,
                                  int, long, int, int, hipStream_t);

// K splits for [N][K] x [M][K]: as many as keep one block on each of the 256
// compute units, with at least 8 steps a split where there are more than four (4
// above 64 rows, where a block has twice the features). A block's ring covers
// the latency by itself, and a second block per unit only added partial sums (us
// with the reduction, 512 / 256 blocks, 24 rows: 4096 x 4096 12.5 / 10.9, K 8192,
// M 2048 14.6 / 12.2, K 4096, M 11008 24.7 / 20.6, M 14336 27.0 / 24.0, 2048 x
// 2048 8.4 / 7.4).
// Up to 64 rows a later count is taken where the units end more evenly, by a
// fifth: K 8192, M 10240 (160 tiles) at 48 rows 47 with 1, 38 with 3; K 3584, M
// 18944 (296) at 1 row 31 with 1, 29 with 2; not from two blocks a unit on (M
// 37888 at 33 rows 56 with 1, 62 with 3). Splits that lie a multiple of 4 KB
// apart fall on the same memory channels as the rows below them: up to twice as
// many are taken if that avoids it as evenly (K 28672, M 8192 at 1 row 90 with 2,
// 77 with 4), or three for four above 64 rows (8192 x 8192 at 72 rows 43.5 /
// 37.4, 128 rows 45 / 43). Up to 64 rows the count does not depend on N, so neither do a row's sums.
extern "C" int ks_skinny_splits(int M, int K, int N, int glu) {
  constexpr int UNITS = 256;
  if (glu) return 1;
  if (ks_mid_takes(M, K, N)) return ks_mid_splits(M, K, N);
  const int bm = feature_tile(N);
  const int tiles = (M + bm - 1) / bm, steps = K / BK;
  if (tiles < 1) return 1;
  int most = steps / 4, s = UNITS / tiles;
  if (N <= 64 && most > 4) most = steps / 8 > 4 ? steps / 8 : 4;
  if (s > most) s = most;
  if (s > 16) s = 16;
  if (s < 1) s = 1;
  if (N > 64) return s == 4 && K % 8192 == 0 ? 3 : s;
  // rounds of blocks on a unit with t splits, each of 1 / t of K
  auto rounds = [&](int t) { return ((long)tiles * t + UNITS - 1) / UNITS; };
  auto aliased = [&](int t) { return K % 2048 == 0 && K * 2L % (t * 4096L) == 0; };
  for (int t = s + 1; tiles < 2 * UNITS && t <= 16 && steps / t >= 12; ++t)
    if (5 * rounds(t) * s <= 4 * rounds(s) * t) {
      s = t;
      break;
    }
  if (s > 1 && aliased(s))
    for (int t = s + 1; t <= 2 * s && t <= 16 && steps / t >= 12; ++t)
      if (!aliased(t) && rounds(t) * s <= rounds(s) * t) return t;
  return s;
}

// `out` null: the sums of the splits stay in `partial` for the caller's kernel. `bias`
// (null: none) is added to the sums in 32 bits; the library copies it into the output
// first at one row (us, K 2048, M 13376 at 1 / 24 / 128 rows 17.5 / 15.3 / 19.6 there, 11.3
// / 11.7 / 18.3 here).
extern "C" hipError_t ks_skinny_gemm(void* out, void* partial, const void* x,
                                     const void* w, const void* bias, int M, int K, int N,
                                     long xs, int splits, int glu, hipStream_t stream) {
  if (N < 1 || N > 256 || M < 1 || M % 4 != 0 || K < BK || K % BK != 0 || splits < 1 ||
      splits > K / BK || ((splits > 1 || !out) && (!partial || glu)) || xs % 8 != 0 ||
      (bias && (glu || !out || M % 8 != 0)) ||
      (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out | (uintptr_t)partial |
        (uintptr_t)bias) & 15) != 0)
    return hipErrorInvalidValue;
  const bool sums = splits > 1 || !out;
  const GemmArgs p{sums ? partial : out, (const short*)x, (const short*)w, M,
                   K, N, xs, 0.f, 0.f, (const short*)bias};
  // (their offsets within a tile are 32 bits wide: longer rows stay here)
  if (!glu && ks_mid_takes(M, K, N) && xs < 1 << 22) {
    const hipError_t e = ks_mid_gemm(p.out, x, w, sums ? nullptr : bias, M, K, N, xs, splits, sums,
                                     stream);
    if (e != hipSuccess) return e;
  } else {
    const int bm = feature_tile(N) / (glu ? 2 : 1);
    const dim3 grid((M + bm - 1) / bm, splits);
#define GO(nt, f, s)                                                           \
  {                                                                            \
    if (glu)                                                                   \
      hipLaunchKernelGGL((skinny_gemm_kernel<nt, f, s, GLU>), grid, dim3(256), \
                         0, stream, p);                                        \
    else if (sums)                                                             \
      hipLaunchKernelGGL((skinny_gemm_kernel<nt, f, s, PARTIAL>), grid,        \
                         dim3(256), 0, stream, p);                             \
    else                                                                       \
      hipLaunchKernelGGL((skinny_gemm_kernel<nt, f, s, BF16_OUT>), grid,       \
                         dim3(256), 0, stream, p);                             \
  }
    FOR_TILE(N, GO)
#undef GO
    HIP_CHECK_KERNEL();
  }
  if (sums && out) {
    const long nm = (long)N * M;
    hipLaunchKernelGGL(reduce_splits_kernel, dim3((unsigned)((nm / 4 + 255) / 256)),
                       dim3(256), 0, stream, (short*)out, (const float*)partial, nm,
                       splits, (const short*)bias, M);
    HIP_CHECK_KERNEL();
  }
  return hipSuccess;
}

// silu-like gate within limits (CLAMPED above), gate and up of w [2 M][K]. The
// activation kernel and its launch take 3.5 us of a decode layer, and the sums reach
// it in 32 bits (hybrid step of 4 layers at 1 / 8 / 24 / 64 sequences 345 -> 342, 380 ->
// 375, 446 -> 435, 652 -> 642 us). Up to 64 rows: above, the library has the product.
extern "C" hipError_t ks_skinny_clamped_glu(void* out, const void* x, const void* w, int M,
                                            int K, int N, long xs, float alpha,
                                            float limit, hipStream_t stream) {
  if (N < 1 || N > 64 || M < 1 || M % 4 != 0 || K < BK || K % BK != 0 || xs % 8 != 0 ||
      (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15) != 0)
    return hipErrorInvalidValue;
  const GemmArgs p{out, (const short*)x, (const short*)w, M, K, N, xs, alpha, limit, nullptr};
  const int bm = feature_tile(N) / 2;
  const dim3 grid((M + bm - 1) / bm, 1);
#define GO(nt, f, s)                                                                     \
  hipLaunchKernelGGL((skinny_gemm_kernel<nt, f, s, CLAMPED>), grid, dim3(256), 0, stream, p);
  FOR_FEW(N, GO)
#undef GO
  HIP_CHECK_KERNEL();
  return hipSuccess;
}
