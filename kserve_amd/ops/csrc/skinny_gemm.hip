// Products of few rows with a weight matrix: out[N][M] = x[N][K] w[M][K]^T for
// N <= 256 tokens (decode batches, short prompts), where reading the weights
// is what bounds them.
//
// A block takes 64 or 128 features and all tokens over a range of K, on the tiles of
// gemm_tile.h: 4 waves (8 above 128 rows), the ring as deep as LDS lets it be (64
// features: two blocks a unit up to 96 rows). K is split over blocks until the chip is
// full; the parts leave fp32 sums that the consumer's kernel or a second one adds in
// order (no atomics). With halves a block's rows are as many gate as up features and
// the activation leaves it directly.
//
// The weights are one bound (6.0 to 6.5 TB/s of rows 128 bytes at a time, K 4096, M
// 28672), the reads of LDS and the products of the few waves of a unit the other: a
// wave that first reads a step's fragments and then multiplies them takes as long for
// both as the weights for their way (36 us of 48 at 96 rows), so the reads and the next
// steps' loads go between the products. us, with a wave's reads ahead of its products
// (and 64 features up to 64 rows, 128 above) / here: K 4096, M 14336 GLU at 1 / 24 / 48 /
// 64 / 96 / 128 / 192 rows 41.0 / 39.7, 42.1 / 40.7, 46.9 / 42.1, 51.0 / 42.8, 48.0 / 45.5, 56.9 /
// 50.9, 74.8 / 60.5 (the library 68.9 and its activation); K 4096, M 32000 at 1 / 64 / 128
// 43.5 / 42.6, 50.7 / 44.4, 60.0 / 54.3; K 14336, M 4096 20.1 / 19.8, 25.0 / 24.5, 31.3 / 28.9;
// K 2048, M 10304 10.3 / 9.3, 15.3 / 13.2, 17.0 / 17.0; K 8192, M 2048 8.0 / 7.7, 9.8 / 9.4,
// 12.7 / 11.9. Token rows straight into registers (sixteen rows to a load, neighbouring
// lanes in different ones) come at a quarter of the rate: 52.9 for 46.9 at 77 rows.
#include "gemm_tile.h"

extern "C" int ks_mid_wide(int, int, int);
extern "C" hipError_t ks_mid_gemm(void*, const void*, const void*, const void*, int, int,
                                  int, long, int, int, int, int, hipStream_t);

namespace {

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

template <int TN, int TM, int WN, int WM, int S, bool LONG = false>
hipError_t go(const DenseArgs& p, int epi, hipStream_t stream) {
  const dim3 grid(p.tiles * p.splits), block(WN * WM * 64);
#define GO(e)                                                                          \
  hipLaunchKernelGGL((dense_gemm_kernel<TN, TM, WN, WM, S, e, true, LONG>), grid, block, \
                     0, stream, p)
  if (epi == GLU) GO(GLU);
  else if (epi == CLAMPED) GO(CLAMPED);
  else if constexpr (TN != 256 || TM != 128) {  // (those of ks_mid_gemm)
    if (epi == PARTIAL) GO(PARTIAL);
    else GO(BIAS);
  }
#undef GO
  HIP_CHECK_KERNEL();
  return hipSuccess;
}

// rows or K of 2^22 elements and more
bool is_long(int K, long xs) { return K >= 1 << 22 || xs >= 1 << 22; }

constexpr int cdiv(long a, long b) { return (int)((a + b - 1) / b); }

// How a product is laid out: which kernel, features of a block, parts of K.
enum Form {
  STREAMED,   // all rows in a block
  ROW_TILES,  // tiles of 128 rows (dense_gemm.hip)
  ONE_PART,   // 97 to 128 rows, 8 waves (dense_gemm.hip)
};
struct Plan {
  Form form;
  int tm, splits;
};

// parts of K that fill the chip with blocks, four steps in each at least
int parts(int tiles, int K) {
  int s = UNITS / tiles;
  if (s > K / BK / 4) s = K / BK / 4;
  return s < 1 ? 1 : s > 16 ? 16 : s;
}

// Up to 64 rows: as many parts as keep one block on each of the 256 compute units,
// with at least 8 steps a part where there are more than four. A second block per unit
// only added partial sums (us with the reduction, 512 / 256 blocks, 24 rows: 4096 x
// 4096 12.5 / 10.9, K 8192, M 2048 14.6 / 12.2, K 4096, M 11008 24.7 / 20.6).
// A later count is taken where the units end more evenly, by a fifth: K 8192, M 10240
// (160 tiles) at 48 rows 47 with 1, 38 with 3; K 3584, M 18944 (296) at 1 row 31 with 1,
// 29 with 2; not from two blocks a unit on (M 37888 at 33 rows 56 with 1, 62 with 3).
// Parts that lie a multiple of 4 KB apart fall on the same memory channels as the rows
// below them: up to twice as many are taken if that avoids it as evenly (K 28672, M
// 8192 at 1 row 90 with 2, 77 with 4). The count does not depend on N, so neither do a
// row's sums.
int few_parts(int M, int K) {
  const int tiles = cdiv(M, 64), steps = K / BK;
  int most = steps / 4, s = UNITS / tiles;
  if (most > 4) most = steps / 8 > 4 ? steps / 8 : 4;
  if (s > most) s = most;
  if (s > 16) s = 16;
  if (s < 1) s = 1;
  // rounds of blocks on a unit with t parts, each of 1 / t of K
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

// A block of 128 features reads the token rows half as often, one of 64 comes to the
// chip's units more evenly and leaves half as many sums.
//
// Up to 64 rows 128 where K is in one part and they fill three quarters of the units'
// rounds, from 17 rows on (us, 64 / 128 features: K 4096, M 28672 at 1 / 24 / 48 / 64
// rows 38.6 / 38.8, 40.0 / 39.1, 44.8 / 40.3, 48.5 / 41.5, M 50304 at 64 89.9 / 82.3;
// but K 2048, M 32000 at 24 / 48 / 64 22.7 / 24.1, 24.8 / 24.6, 26.3 / 25.0).
//
// Above by an estimate from the times of K 1024 to 14336, M 1024 to 50304 (weights not in a
// cache): a launch, the steps of the busiest unit and the sums that are written, off by 5 %
// in the mean (K 14336, M 4096 at 96 / 256 rows 27.6 / 25.6, 53.6 / 38.6; K 4096, M 4096 10.4
// / 11.8, 18.3 / 21.4, M 6144 15.9 / 14.4, 27.0 / 23.7; K 2048, M 16384 16.5 / 23.9, 26.7 /
// 35.6); in parts no caller's K is shorter (gate|up to 112 rows: M 12288 to 16384, K 64 to
// 960 15 % ahead of the kernel before in the mean, 2 % behind at most). Past 8192 features a
// pass of its own adds the sums, to 10240 features the norm's kernel for some callers: those
// cost less (one part of 64 features / three of 128, with the norm: K 3072, M 10240 at 65 /
// 160 / 192 rows 26.9 / 23.8, 37.0 / 29.8, 39.8 / 31.1, without at 192 32.8 / 29.5; K 2048 at
// 65 / 129 19.3 / 21.7, 23.8 / 27.5).
//
// To 128 rows, 8192 features and K 8192 parts of 128 features cost 2.25 us more, since they
// leave twice as many sums to add (us, 128 features / 64, with the norm that adds them: M
// 6144, K 3776 at 70 / 96 / 127 rows 20.8 / 18.9, 22.8 / 20.3, 25.9 / 23.2, K 4608 22.3 /
// 21.1, 24.4 / 23.2, 27.4 / 26.2; M 4776, K 7168 24.9 / 22.7, 26.4 / 24.2 at 84, 29.9 / 27.6;
// M 5120, K 8192 at 128 31.8 / 28.8; not K 6144, M 7168 at 127 32.9 / 35.0): over K 2048 to
// 8192, M 2112 to 8192 0.1 % off the better one, 1.4 % without. On longer K it is the other
// way in a model (a 77-token prompt of 4 layers 504, with K 14336 so too 516).
//
// At 129 to 192 rows blocks of 64 features fall behind where K is long: in more than two parts
// from token rows of 1.6 MB on, in two of 1.4, in one part from K 3840 on, but where the
// other's two parts lie a multiple of 4 KB apart (us, 64 features / 128, with the sums added:
// M 13824, K 3584 at 160 / 176 rows 34.2 / 35.7, 36.3 / 37.7, K 4608 43.3 / 41.8, 46.4 /
// 43.3, K 5120 52.9 / 45.7, 53.9 / 46.7, but M 16384, K 4096 at 176 38.5 / 40.9; M 4352, K
// 4096 at 160 / 192 21.4 / 22.8, 23.7 / 24.1, K 5120 at 160 / 176 26.0 / 23.8, 27.8 / 24.7; M
// 7168, K 4096 at 176 / 192 28.1 / 25.9, 29.6 / 26.7; M 5120, K 6144 29.9 / 26.5, 30.1 /
// 27.6). Over K 2112 to 8192 and M 4352 to 16384 this takes the better one to 0.1 % in the
// mean, to 4 % without.
Plan plan(int M, int K, int N, bool halves) {
  const long rows = halves ? 2L * M : M;
  const int tiles = cdiv(rows, 128), steps = K / BK;
  if (N <= 64) {
    const int s = halves ? 1 : few_parts(M, K);
    const bool even = 4L * tiles >= 3L * UNITS * cdiv(tiles, UNITS);
    return {STREAMED, s == 1 && even && (N > 32 || (N > 16 && K >= 4096)) ? 128 : 64, s};
  }
  if (!halves && ks_mid_wide(M, K, N)) return {N > 96 ? ONE_PART : STREAMED, 64, 1};
  // Small weights: their rows twice rather than all token rows in a block (us, K 2048, M
  // 2048 at 129 / 192 / 256 rows 7.4 / 8.8 / 10.1 streamed, 7.7 / 7.8 / 7.8 so, M 4096 9.4 / 10.9
  // / 12.9, 11.3 / 11.4 / 11.8), and above 192 rows some larger ones, which leave half as
  // many sums to add (with those, K 8192, M 2048 at 193 / 224 / 256 21.5 / 23.4 / 25.3
  // streamed, 20.6 / 20.7 / 21.1 so, added by the norm K 2048, M 4096 at 193 / 224 18.7 /
  // 19.9, 15.6 / 15.9, K 3072 at 224 22.4, 20.0; K 8192, M 2560 at 224, sums, added by a
  // pass, by the norm 18.9, 28.5, 28.8 streamed, 21.1, 24.2, 25.1 so, M 2112 17.7, 22.0, 23.2
  // and 21.0, 23.6, 25.0 at 193; but K 4096, M 3072 without at 224 15.8, 18.1).
  if (!halves && N > 128 && M <= 4096 &&
      ((long)K * M <= 3000000 + (N - 128) * 50000L ||
       (N > 192 && (M <= 2048 || (M > 2240 && M <= 2560 && K > 7168) ? K <= 8192
                                                                       : M > 3584 && K <= 3072)))) {
    const int n = 2 * cdiv(M, 64);
    return {ROW_TILES, 64, parts(n, K)};
  }
  static constexpr struct {
    float launch[2], step[2];  // us, of 64 and 128 features
    float sums;                // per MB
  } COST[4] = {{{0.f, 2.f}, {0.44f, 0.65f}, 0.45f},
               {{0.f, 0.f}, {0.46f, 0.72f}, 0.5f},
               {{0.f, 2.f}, {0.58f, 0.79f}, 0.4f},
               {{0.f, 0.5f}, {0.8f, 0.92f}, 0.5f}};
  const auto& cost = COST[N <= 96 ? 0 : N <= 128 ? 1 : N <= 192 ? 2 : 3];
  const bool long_k = !halves && N > 128 && N <= 192 && M > 4096;
  Plan best{STREAMED, 64, 1};
  float least = 0.f;
  for (int i = 0; i < 2; ++i) {
    const int tm = 64 << i, n = cdiv(rows, tm), s = halves ? 1 : parts(n, K);
    const float us = cost.launch[i] +
                     cost.step[i] * (cdiv(steps, s) * (float)cdiv((long)n * s, UNITS)) +
                     (s > 1 ? cost.sums * 4e-6f * s * N * M : 0.f) +
                     (s > 1 && M > 8192 ? M > 10240 ? 6.f : 2.5f : 0.f) +
                     (i == 1 && s > 1 && N <= 128 && M <= 8192 && K <= 8192 ? 2.25f : 0.f) +
                     (i == 0 && long_k &&
                              (s > 1 ? (long)N * K > (s > 2 ? 800000 : 700000)
                                     : K >= 3840 && K % 4096 != 0)
                          ? 8.f
                          : 0.f);
    if (i == 0 || us < least) {
      least = us;
      best = {STREAMED, tm, s};
    }
  }
  return best;
}

// Whether an XCD takes all parts of its features (gemm_tile.h): where 2.5 MB of token rows and
// its share of the sums fit its L2 of 4 MB (us with the sums added, else / so: K 8192, M 8192
// at 129 / 256 rows 39.4 / 36.4, 47.1 / 52.0, K 14336, M 5120 at 192 44.5 / 58.6; K 8192, M
// 9216 at 160 43.1 / 45.6). Up to 128 rows the sums are few. Every eighth block above 192
// rows to K 10240, past which it is level, but where parts lie powers of two apart (at 193
// rows, runs / in turn, K 7168, M 5120 32.9 / 30.5, K 8064 34.2 / 31.9, K 10240 39.3 / 37.3,
// K 8192, M 4352 32.7 / 34.8, M 9728 50.0 / 50.5).
Order order(int M, int K, int N) {
  if (N > 128 && M <= 8192 && (long)N * K <= 5 << 18) return PARTS_FIRST;
  return N > 192 && K <= 10240 && K != 8192 ? IN_TURN : RUNS;
}

hipError_t run(DenseArgs p, int tm, int epi, hipStream_t stream) {
  const bool far = is_long(p.K, p.long_xs);
  if (far) tm = 64;
  const int tf = has_halves(epi) ? tm / 2 : tm;
  const long tiles = ((long)p.M + tf - 1) / tf;
  // (HIP's most threads)
  if (tiles * p.splits * (p.N > 128 ? 512 : 256) >= 1L << 32) return hipErrorInvalidValue;
  p.ftiles = p.tiles = (int)tiles;
  const int N = p.N;
  if (far)
    return N <= 64 ? go<64, 64, 2, 2, 5, true>(p, epi, stream)
                   : go<256, 64, 4, 2, 4, true>(p, epi, stream);
  if (tm == 64)
    return N <= 32    ? go<32, 64, 2, 2, 6>(p, epi, stream)
           : N <= 64  ? go<64, 64, 2, 2, 5>(p, epi, stream)
           : N <= 96  ? go<96, 64, 2, 2, 4>(p, epi, stream)
           : N <= 128 ? go<128, 64, 2, 2, 4>(p, epi, stream)
           : N <= 192 ? go<192, 64, 4, 2, 5>(p, epi, stream)
                      : go<256, 64, 4, 2, 4>(p, epi, stream);
  if (N > 192 && !has_halves(epi))
    return ks_mid_gemm(p.out, p.x, p.w, p.bias, p.M, p.K, N, p.long_xs, p.splits, epi == PARTIAL, 128,
                       p.order, stream);
  return N <= 32    ? go<32, 128, 2, 2, 7>(p, epi, stream)
         : N <= 64  ? go<64, 128, 2, 2, 6>(p, epi, stream)
         : N <= 96  ? go<96, 128, 2, 2, 5>(p, epi, stream)
         : N <= 128 ? go<128, 128, 2, 2, 5>(p, epi, stream)
         : N <= 192 ? go<192, 128, 4, 2, 4>(p, epi, stream)
                    : go<256, 128, 4, 2, 3>(p, epi, stream);
}

}  // namespace

extern "C" int ks_skinny_splits(int M, int K, int N, int glu) {
  return M < 1 ? 1 : plan(M, K, N, glu).splits;
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
  const DenseArgs p{sums ? partial : out, (const short*)x, (const short*)w,
                    (const short*)(sums ? nullptr : bias), M, K, N, (int)xs, 0, 0, splits,
                    order(M, K, N), 0.f, 0.f, xs};
  const Plan how = plan(M, K, N, glu);
  const hipError_t err =
      how.form != STREAMED && !is_long(K, xs)
          ? ks_mid_gemm(p.out, x, w, p.bias, M, K, N, xs, splits, sums, 64, RUNS, stream)
          : run(p, how.tm, glu ? GLU : sums ? PARTIAL : BIAS, stream);
  if (err != hipSuccess) return err;
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
// 375, 446 -> 435, 652 -> 642 us).
extern "C" hipError_t ks_streamed_clamped_glu(void* out, const void* x, const void* w,
                                              int M, int K, int N, long xs, float alpha,
                                              float limit, hipStream_t stream) {
  if (N < 1 || N > 256 || M < 1 || M % 4 != 0 || K < BK || K % BK != 0 || xs % 8 != 0 ||
      (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15) != 0)
    return hipErrorInvalidValue;
  return run({out, (const short*)x, (const short*)w, nullptr, M, K, N, (int)xs, 0, 0, 1,
              RUNS, alpha, limit, xs},
             plan(M, K, N, true).tm, CLAMPED, stream);
}
