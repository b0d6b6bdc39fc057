// Products of an encoder's layers: out[N][M] = act(x[N][K] w[M][K]^T + bias), bf16
// with fp32 sums, act the identity or gelu (erf form) on the fp32 sums.
//
// K is short here (768: twelve steps), so a tile's first loads, its epilogue and
// the last, uneven round of tiles weigh as much as the products, and the library,
// whose choice of tile changes from one token count to the next, ran at 0.4 to 0.9
// PFLOP/s with a pass over memory of its own for gelu. Each step's token and
// weight rows come by LDS-direct loads into one slot of a ring; a wave reads the
// fragments of a half step while it multiplies those of the half before, with one
// barrier per step, and its reads and loads go between the products. Where a unit
// has one block, LDS bounds it: 128 bytes a cycle for reads and loads (128 x 192 in
// 8 waves: 1344 cycles a step, 768 of them products; 1310 measured, 1400 with the
// reads and loads in a row). Where it has two, the latency of the one step that two
// slots hold in flight does (1.7 us a step of both); 32-wide steps in four slots took
// 41 us for 34, their 64-byte rows come at two thirds of the rate. The rows of a
// fragment never share a bank (0 conflicts).
//
// us, this / the library (and gelu's kernel): 7864 x 768 to 2304 32 / 63, to 768
// 12.6 / 15.1, to 3072 with gelu 44 / 68; 7864 x 3072 to 768 32 / 40; 1500 rows to 768 7.0
// / 8.7, to 3072 with gelu 14.6 / 20.9; 200 rows to 2304 5.4 / 7.9.
#include "gemm_tile.h"

namespace {

// Which tile: the least a n + b, for n tiles on the busiest unit (a quarter more for
// an odd one where two blocks share a unit: alone it hides less of its latency). a
// and b are us at K 768 without gelu, fitted over 768 to 3072 features and 1200 to
// 12000 rows; all grow with K and gelu alike, so the order holds but for the largest tile,
// whose one round has nothing to hide its first loads and its output behind: on short K
// it is not taken (us, tiles of 128 x 128 / so, at K 128, 256, 384, 512, 640, 768, 1024, 1536:
// 8086 x K to 1896 11.2 / 12.9, 15.4 / 15.9, 18.2 / 20.9, 21.6 / 23.9, 26.1 / 26.5, 29.3 / 29.5,
// 34.6 / 35.3, 49.2 / 46.7; 2886 to 2312 7.4 / 8.4, 8.9 / 9.7, 10.9 / 11.2, 12.6 / 12.9, 14.5 /
// 14.0, 16.1 / 16.2, 19.6 / 18.4, 26.7 / 23.9; with gelu 4800 to 3072 15.9 / 17.7, 19.1 / 21.2,
// 22.5 / 24.4, 25.7 / 26.9, 29.3 / 30.6, 33.2 / 33.7, 39.6 / 39.0, 54.8 / 50.5; than tiles of 64 x 128 it is better from K
// 512 on, 5429 to 1024 12.0 / 11.1, 3034 to 2048 13.1 / 12.5). Where a unit has a
// single tile, one block of eight waves with a deeper ring beats one of four (7864 x
// 768 to 768 13.5 / 15.0, 1200 to 2304 10.5 / 12.8). The largest tile is for what it
// alone brings into one round (us, without / with it: 9000 x 768 to 768 15.7 / 14.7, 2048
// to 768 28.5 / 26.5, 3072 to 768 43.0 / 38.3, 5400 x 3072 to 1024 46 / 31.8, 8000 57 / 42, 8000
// x 4096 to 1024 63 / 55).
struct Tile {
  int tn, tm;
  float a, b;
  bool pairs;
};
constexpr int NTILES = 7, LARGEST = 6;
constexpr Tile TILES[NTILES] = {
    {128, 192, 12.6f, 0.5f, false}, {128, 192, 9.8f, 2.f, true},
    {128, 128, 9.5f, 0.f, false},   {128, 128, 7.2f, 2.2f, true},
    {64, 128, 4.4f, 2.6f, false},   {64, 64, 2.9f, 2.5f, false},
    {256, 128, 14.1f, 0.5f, false}};

}  // namespace

extern "C" int ks_dense_tile(int M, int N, int K) {
  int best = 0;
  float least = 0.f;
  for (int i = 0; i < NTILES; ++i) {
    if (i == LARGEST && K < (TILES[best].pairs ? 704 : 512)) continue;
    const Tile& t = TILES[i];
    const long tiles = (long)((M + t.tm - 1) / t.tm) * ((N + t.tn - 1) / t.tn);
    const long n = (tiles + UNITS - 1) / UNITS;
    const float us = t.a * ((float)n + (t.pairs && n % 2 ? 0.25f : 0.f)) + t.b;
    if (i == 0 || us < least) {
      least = us;
      best = i;
    }
  }
  return best;
}

// `tile` < 0: by the rule above
extern "C" hipError_t ks_dense_gemm(void* out, const void* x, const void* w,
                                    const void* bias, int M, int K, int N, long xs,
                                    int gelu, int tile, hipStream_t stream) {
  // (rows within a tile and steps along K by 32-bit offsets)
  if (N < 1 || M < 8 || M % 8 != 0 || K < BK || K % BK != 0 || K >= 1 << 22 ||
      xs % 8 != 0 || xs < K || xs >= 1 << 22 || tile >= NTILES ||
      (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out | (uintptr_t)bias) & 15) != 0)
    return hipErrorInvalidValue;
  if (tile < 0) tile = ks_dense_tile(M, N, K);
  const Tile& t = TILES[tile];
  const long ftiles = (M + t.tm - 1) / t.tm, tiles = ftiles * ((N + t.tn - 1) / t.tn);
  if (tiles > 0x7fffffff) return hipErrorInvalidValue;
  const DenseArgs p{out, (const short*)x, (const short*)w, (const short*)bias,
                    M, K, N, (int)xs, (int)ftiles, (int)tiles, 1, 0, 0.f, 0.f, xs};
#define GO(tn, tm, wn, wm, s)                                                         \
  if (gelu)                                                                           \
    hipLaunchKernelGGL((dense_gemm_kernel<tn, tm, wn, wm, s, BIAS_GELU>),             \
                       dim3(p.tiles), dim3(wn * wm * 64), 0, stream, p);              \
  else                                                                                \
    hipLaunchKernelGGL((dense_gemm_kernel<tn, tm, wn, wm, s, BIAS>), dim3(p.tiles),   \
                       dim3(wn * wm * 64), 0, stream, p);
  switch (tile) {
    case 0: GO(128, 192, 4, 2, 3) break;
    case 1: GO(128, 192, 2, 2, 2) break;
    case 2: GO(128, 128, 4, 2, 4) break;
    case 3: GO(128, 128, 2, 2, 2) break;
    case 4: GO(64, 128, 2, 2, 3) break;
    case 5: GO(64, 64, 2, 2, 4) break;
    default: GO(256, 128, 4, 2, 3) break;
  }
#undef GO
  HIP_CHECK_KERNEL();
  return hipSuccess;
}

// Wide products of 65 to 128 rows in one round of blocks of 64 features and all rows, K in
// one part: from 97 rows on 8 waves here, below on the streaming tiles of 96 rows
// (skinny_gemm.hip). Bound by the reads of W and, per unit, as many of x. us, so / the
// library at 65, 96 and 128 rows, weights not in a cache: K 1024, M 10304 8.5 / 13.1, 9.3 /
// 13.5, 10.4 / 14.1; K 2048, M 10304 13.7 / 21.4, 15.1 / 17.7, 17.0 / 18.9, M 16384 15.0 /
// 19.2, 16.4 / 19.9, 18.0 / 21.0; K 3072, M 16384 21.4 / 25.7, 23.4 / 27.8, 27.7 / 29.6; K
// 4096, M 14336 24.6 / 31.6, 27.2 / 33.3, 30.9 / 35.0. The lines are from a kernel before, of
// which these were ahead by a tenth to a half: not past K 4608, where that turned (K 5120, M
// 12288 at 65 / 112 rows 32.1 / 33.9, 37.5 / 39.9, M 16384 at 128 43.9 / 44.9), nor where K is
// long and a quarter of the units idle (K 4096, M 10304 23.8 / 22.4, 28.2 / 28.4); past 256
// tiles a second round is nearly empty (K 2048, M 17408 26.4 / 23.3); the line at 129 tiles is
// from weights that came through the caches (K 2048, M 8192 at 128 rows 16.9, library 15.7,
// as they are loaded now 14.8), and it could be lower.
static bool mid_wide(int M, int K, int N) {
  const int tiles = (M + 63) / 64;
  return N > 64 && N <= 128 && tiles <= UNITS && K >= 512 && K <= 4608 &&
         (K <= 2048 ? tiles > 128 : tiles >= 192);
}
extern "C" int ks_mid_wide(int M, int K, int N) { return mid_wide(M, K, N); }

// Forms of the few-row products (skinny_gemm.hip): tiles of 128 rows and 64 features
// for small weights, K in parts, and for the wide products above; 128 features of all
// of 193 to 256 rows. out: fp32 sums of the parts (sums) or bf16 with the bias, if there
// is one
extern "C" hipError_t ks_mid_gemm(void* out, const void* x, const void* w,
                                  const void* bias, int M, int K, int N, long xs,
                                  int splits, int sums, int tm, int order,
                                  hipStream_t stream) {
  if ((bias && (sums || M % 8 != 0)) || N < 1 || N > 256 || M < 4 || M % 4 != 0 || K < BK || K % BK != 0 ||
      K >= 1 << 22 || xs % 8 != 0 || xs >= 1 << 22 || splits < 1 || splits > K / BK ||
      (splits > 1 && !sums) ||
      (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out | (uintptr_t)bias) & 15) != 0)
    return hipErrorInvalidValue;
  DenseArgs p{out, (const short*)x, (const short*)w, (const short*)bias, M, K, N, (int)xs,
              0, 0, splits, order, 0.f, 0.f, xs};
#define GO(tn, tm, wn, wm, s, epi, stream_)                                           \
  {                                                                                   \
    p.ftiles = (M + tm - 1) / tm;                                                     \
    p.tiles = p.ftiles * ((N + tn - 1) / tn);                                         \
    hipLaunchKernelGGL((dense_gemm_kernel<tn, tm, wn, wm, s, epi, stream_>),          \
                       stream_ ? dim3(p.tiles * splits) : dim3(p.tiles, splits),      \
                       dim3(wn * wm * 64), 0, stream, p);                             \
  }
  if (tm == 64) {
    if (sums) GO(128, 64, 2, 2, 3, PARTIAL, false)
    else GO(128, 64, 4, 2, 4, BIAS, false)
  } else {
    if (sums) GO(256, 128, 4, 2, 3, PARTIAL, true)
    else GO(256, 128, 4, 2, 3, BIAS, true)
  }
#undef GO
  HIP_CHECK_KERNEL();
  return hipSuccess;
}
