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
// 12.6 / 15.1, to 3072 with gelu 44 / 68; 1500 rows to 768 7.0 / 8.7, to 3072 with
// gelu 14.6 / 20.9; 200 rows to 2304 5.4 / 7.9.
#include "common.h"
#include "mfma_layouts.h"

namespace {

constexpr int UNITS = 256;  // compute units
constexpr int BK = 64;  // K per step

// sums + bias in bf16; gelu of it; fp32 sums of the K splits
enum Epilogue { BIAS, BIAS_GELU, PARTIAL };

struct DenseArgs {
  void* out;          // [N][M] bf16; PARTIAL: [splits][N][M] fp32
  const short* x;     // [N][K], row stride xs
  const short* w;     // [M][K]
  const short* bias;  // [M] or null
  int M, K, N, xs;
  int ftiles, tiles;  // tiles along M, in all
};

typedef __attribute__((address_space(3))) void lds_t;

// 16 bytes per lane from a uniform address (lane and step offsets below 2^32)
// straight to 1 KB of LDS
constexpr int NT_AUX = 2;  // cache policy of a non-temporal load
template <int AUX = 0>
__device__ __forceinline__ void load_lds(const short* from, short* to, unsigned int lane_at,
                                         int step_at) {
  const __amdgpu_buffer_rsrc_t rows =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<short*>(from), 0, -1, 0x00027000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, (lds_t*)to, 16, lane_at, step_at, 0, AUX);
}

// s_waitcnt with vmcnt <= n (bits 3:0 and 15:14), lgkmcnt 0, expcnt free
constexpr int wait_imm(int n) { return (0x7 << 4) | (n & 0xF) | ((n >> 4) << 14); }

// x Phi(x) with the tail Phi(-|x|) = exp(-x^2 / 2) t Q(t), t = 1 / (1 + c |x|), Q a
// polynomial fitted to a relative 6.5e-7 of it over |x| < 13.4 (least squares,
// reweighted towards the largest error): a third of erff's instructions, which
// would cost as much as the products.
__device__ __forceinline__ float gelu_f(float x) {
  const float a = fabsf(x);
  const float t = __builtin_amdgcn_rcpf(1.f + 0.265165043f * a);
  float q = -0.0675466018f;
  q = q * t + 0.193964045f;
  q = q * t - 0.0647915465f;
  q = q * t + 0.141525405f;
  q = q * t + 0.0833345009f;
  q = q * t + 0.107844114f;
  q = q * t + 0.105669766f;
  const float tail = q * t * __builtin_amdgcn_exp2f(x * x * -0.721347520f);
  return x * (x > 0.f ? 1.f - tail : tail);
}

template <int TN, int TM, int WN, int WM, int S, int EPI>
__global__ __launch_bounds__(WN * WM * 64, 2) void dense_gemm_kernel(const DenseArgs p) {
  constexpr int NW = WN * WM;
  constexpr int FN = TN / WN / 16, FM = TM / WM / 16;  // fragments of a wave
  constexpr int STAGE = (TN + TM) * BK;                // elements
  constexpr int NX = TN / 8 / NW, NI = (TN + TM) / 8 / NW;  // 1 KB loads of a wave
  constexpr int LAG = (FM + FN) / 2;  // a half step's reads end by 2/3 of its products
  constexpr int N1 = S == 2 ? NI : (NI + 1) / 2;  // of them, right after the barrier
  static_assert(TN % (8 * NW) == 0 && TM % (8 * NW) == 0 && FM % 2 == 0 && S >= 2 &&
                    S * STAGE * 2 <= 160 * 1024,
                "tile");
  __shared__ __attribute__((aligned(16))) short ring[S * STAGE];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, g = lane >> 4;

  // blocks go to the 8 XCDs in turn: each takes a run of tiles, features first
  const int xcd = blockIdx.x & 7, nth = blockIdx.x >> 3;
  const int tile = xcd * (p.tiles >> 3) + min(xcd, p.tiles & 7) + nth;
  const int n0 = tile / p.ftiles * TN, m0 = tile % p.ftiles * TM;
  const int all = p.K / BK;
  const int lo = (int)((long)all * blockIdx.y / gridDim.y);  // of this K split
  const int steps = (int)((long)all * (blockIdx.y + 1) / gridDim.y) - lo;

  // a load is 8 rows of 128 bytes; 16-byte chunk c of a row sits at c ^ key, the
  // key such that the rows of a fragment at one chunk hit different banks
  const short* xb = p.x + (long)n0 * p.xs + lo * BK;
  const short* wb = p.w + (long)m0 * p.K + lo * BK;
  unsigned int at[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int r = ((i < NX ? i : i - NX) * NW + wave) * 8 + (lane >> 3);
    const int key = i < NX ? (r >> 1) & 7 : ((r >> 1) & 1) | ((r >> 2) & 6);
    const unsigned int row =
        i < NX ? min(r, p.N - 1 - n0) * p.xs : min(r, p.M - 1 - m0) * p.K;
    at[i] = (row + ((lane & 7) ^ key) * 8) * 2;
  }
  // Wide products of few rows start their blocks' steps apart, as the few-row kernel
  // does: rows of W a multiple of 4 KB apart would keep all blocks on the same memory
  // channels (us at 128 rows of K 2048, M 16384 19.1 -> 18.3, of K 4096 34.7 -> 32.5)
  constexpr bool APART = TN == 128 && TM == 64 && EPI == BIAS;
  const int rot = APART ? (int)(blockIdx.x >> 1) % steps : 0;
  auto issue = [&](int step, int slot, int i) {
    if constexpr (APART) {
      step += rot;
      step -= step >= steps ? steps : 0;
    }
    short* const to = &ring[slot * STAGE + (i * NW + wave) * 8 * BK];
    // Weights that one block alone reads pass the caches by: they leave no room there
    // otherwise to what the next kernels read and to what the last ones wrote (steps in
    // us: hybrid 72 / 128 sequences 695 -> 683, 992 -> 981, llama 256 2268 -> 2260, 192
    // level). Not the narrow products' in parts (72 / 128 sequences 8 and 6 us slower).
    if ((APART || TN == 256) && i >= NX) load_lds<NT_AUX>(wb, to, at[i], step * BK * 2);
    else load_lds(i < NX ? xb : wb, to, at[i], step * BK * 2);
  };

  const int wn = wave % WN, wm = wave / WN;
  f32x4_t acc[FM][FN];
#pragma unroll
  for (int f = 0; f < FM; ++f)
#pragma unroll
    for (int t = 0; t < FN; ++t) acc[f][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // fragment rows: tokens in order; features so that a lane's rows of two
  // fragments are 8 consecutive ones, 16 bytes of the output
  const int xrow = wn * FN * 16 + col, xkey = (col >> 1) & 7;
  const int frow = TN + wm * FM * 16 + (col >> 2) * 8 + (col & 3);
  const int fkey = ((col >> 1) & 1) | ((col >> 2) << 1);

  bf16x8_t a0[FM], b0[FN], a1[FM], b1[FN];  // the two halves of a step
  auto fetch_one = [&](int slot, int half, bf16x8_t(&a)[FM], bf16x8_t(&b)[FN], int i) {
    const short* st = &ring[slot * STAGE];
    const short* fp = st + frow * BK + ((half * 4 + g) ^ fkey) * 8;
    const short* xp = st + xrow * BK + ((half * 4 + g) ^ xkey) * 8;
    if (i >= 1 && i <= FM)
      a[i - 1] = *reinterpret_cast<const bf16x8_t*>(
          fp + (((i - 1) >> 1) * 32 + ((i - 1) & 1) * 4) * BK);
    else
      b[i ? i - FM : 0] =
          *reinterpret_cast<const bf16x8_t*>(xp + (i ? i - FM : 0) * 16 * BK);
  };
  auto fetch = [&](int slot, int half, bf16x8_t(&a)[FM], bf16x8_t(&b)[FN]) {
#pragma unroll
    for (int i = 0; i < FM + FN; ++i) fetch_one(slot, half, a, b, i);
    __builtin_amdgcn_sched_barrier(0);
  };
  // A half step's products, between them the reads of the next half step and loads
  // first .. last - 1 of a step to come: a wave that issues those in a row waits for
  // each to be taken while its matrix core idles.
  auto multiply = [&](bf16x8_t(&a)[FM], bf16x8_t(&b)[FN], bf16x8_t(&an)[FM],
                      bf16x8_t(&bn)[FN], int slot, int half, int step, int free_slot,
                      int first, int last) {
    constexpr int T = FM * FN;
#pragma unroll
    for (int t = 0; t < FN; ++t)
#pragma unroll
      for (int f = 0; f < FM; ++f) {
        const int m = t * FM + f;
        acc[f][t] = mfma16x16x32(a[f], b[t], acc[f][t]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < FM + FN; ++i)
          if (i * T / (FM + FN + LAG) == m) fetch_one(slot, half, an, bn, i);
#pragma unroll
        for (int i = first; i < last; ++i)
          if (m == (i - first) * T / (last > first ? last - first : 1))
            issue(step, free_slot, i);
        __builtin_amdgcn_sched_barrier(0);
      }
  };
  auto barrier = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  const bool ring_full = steps >= S;
#pragma unroll
  for (int j = 0; j < S; ++j)
#pragma unroll
    for (int i = 0; i < NI; ++i)
      if (j < steps && (i < N1 || j < S - 1)) issue(j, j, i);
  if (ring_full) __builtin_amdgcn_s_waitcnt(wait_imm(NI * (S - 2) + N1));
  else __builtin_amdgcn_s_waitcnt(wait_imm(0));
  barrier();
  fetch(0, 0, a0, b0);
  // In a step, this wave has read all of it and its own loads of the next have
  // landed before the barrier, which covers the other waves'; then the slot is
  // free. (A loop of its own for the steps that load no more: with the loads under
  // a condition the compiler moves every accumulator once a step.)
  int slot = 0, before = S - 1, j = 0;
  for (; j + S < steps; ++j) {
    multiply(a0, b0, a1, b1, slot, 1, j + S - 1, before, N1, NI);
    __builtin_amdgcn_s_waitcnt(wait_imm(NI * (S - 2)));
    barrier();
    before = slot;
    slot = slot + 1 == S ? 0 : slot + 1;
    multiply(a1, b1, a0, b0, slot, 0, j + S, before, 0, N1);
  }
  if (ring_full)
#pragma unroll
    for (int i = N1; i < NI; ++i) issue(j + S - 1, before, i);
  for (; j + 1 < steps; ++j) {
    multiply(a0, b0, a1, b1, slot, 1, 0, 0, 0, 0);
    __builtin_amdgcn_s_waitcnt(wait_imm(0));
    barrier();
    slot = slot + 1 == S ? 0 : slot + 1;
    multiply(a1, b1, a0, b0, slot, 0, 0, 0, 0, 0);
  }
  // This lane's bias, under the last step's products: in the epilogue each would be
  // waited for, and with it the stores of the features before, since loads and stores
  // count as one (us, 7864 rows: 768 to 2304 32.4 -> 31.8, to 3072 with gelu 51 -> 46, to
  // 768 12.8 -> 12.4; 1500 rows with gelu 15.5 -> 14.3). No earlier: the ring's waits
  // count loads.
  short8_t bias[FM / 2];
#pragma unroll
  for (int f = 0; f < FM; f += 2) {
    const int feat = m0 + wm * FM * 16 + f * 16 + g * 8;
    bias[f / 2] = short8_t{};
    if (EPI != PARTIAL && p.bias && feat < p.M)
      bias[f / 2] = *reinterpret_cast<const short8_t*>(p.bias + feat);
  }
  __builtin_amdgcn_sched_barrier(0);
  multiply(a0, b0, a1, b1, slot, 1, 0, 0, 0, 0);
#pragma unroll
  for (int t = 0; t < FN; ++t)
#pragma unroll
    for (int f = 0; f < FM; ++f) acc[f][t] = mfma16x16x32(a1[f], b1[t], acc[f][t]);
  if constexpr (EPI != PARTIAL) {  // (left to itself the compiler loads it at its use)
#pragma unroll
    for (int f = 0; f < FM / 2; ++f) asm volatile("" : "+v"(bias[f]));
  }

#pragma unroll
  for (int f = 0; f < FM; f += 2) {
    const int feat = m0 + wm * FM * 16 + f * 16 + g * 8;
    if (feat >= p.M) continue;
    if constexpr (EPI == PARTIAL) {
#pragma unroll
      for (int t = 0; t < FN; ++t) {
        const int tok = n0 + wn * FN * 16 + t * 16 + col;
        if (tok >= p.N) continue;
        f32x4_t* o = reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(p.out) +
                                                ((long)blockIdx.y * p.N + tok) * p.M + feat);
        o[0] = acc[f][t];
        if (feat + 4 < p.M) o[1] = acc[f + 1][t];
      }
    } else {
      float b[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) b[r] = bf16_bits_to_float(bias[f / 2][r]);
#pragma unroll
      for (int t = 0; t < FN; ++t) {
        const int tok = n0 + wn * FN * 16 + t * 16 + col;
        if (tok >= p.N) continue;
        bf16x8_t o;
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          float v = acc[f + r / 4][t][r % 4] + b[r];
          if constexpr (EPI == BIAS_GELU) v = gelu_f(v);
          o[r] = (__bf16)v;
        }
        short* to = reinterpret_cast<short*>(p.out) + (long)tok * p.M + feat;
        if (p.M % 8 == 0) {
          // (as wide as these are, they are no longer in the L2 when the next product
          // reads them, and leave it to this one's operands: us, 7864 rows 768 to 3072
          // 47.2 -> 43.7; without gelu attention and norms lose what this gains)
          if constexpr (EPI == BIAS_GELU)
            __builtin_nontemporal_store(o, reinterpret_cast<bf16x8_t*>(to));
          else
            *reinterpret_cast<bf16x8_t*>(to) = o;
        } else {  // (M a multiple of 4)
          typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
          *reinterpret_cast<bf16x4_t*>(to) = bf16x4_t{o[0], o[1], o[2], o[3]};
          if (feat + 4 < p.M)
            *reinterpret_cast<bf16x4_t*>(to + 4) = bf16x4_t{o[4], o[5], o[6], o[7]};
        }
      }
    }
  }
}

// Which tile: the least a n + b, for n tiles on the busiest unit (a quarter more for
// an odd one where two blocks share a unit: alone it hides less of its latency). a
// and b are us at K 768 without gelu, fitted over 768 to 3072 features and 1200 to
// 12000 rows; all grow with K and gelu alike, so the order holds. Where a unit has a
// single tile, one block of eight waves with a deeper ring beats one of four (7864 x
// 768 to 768 13.5 / 15.0, 1200 to 2304 10.5 / 12.8).
struct Tile {
  int tn, tm;
  float a, b;
  bool pairs;
};
constexpr int NTILES = 6;
constexpr Tile TILES[NTILES] = {
    {128, 192, 12.6f, 0.5f, false}, {128, 192, 9.8f, 2.f, true},
    {128, 128, 9.5f, 0.f, false},   {128, 128, 7.2f, 2.2f, true},
    {64, 128, 4.4f, 2.6f, false},   {64, 64, 2.9f, 2.5f, false}};

}  // namespace

extern "C" int ks_dense_tile(int M, int N) {
  int best = 0;
  float least = 0.f;
  for (int i = 0; i < NTILES; ++i) {
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
  if (tile < 0) tile = ks_dense_tile(M, N);
  const Tile& t = TILES[tile];
  const long ftiles = (M + t.tm - 1) / t.tm, tiles = ftiles * ((N + t.tn - 1) / t.tn);
  if (tiles > 0x7fffffff) return hipErrorInvalidValue;
  const DenseArgs p{out, (const short*)x, (const short*)w, (const short*)bias,
                    M, K, N, (int)xs, (int)ftiles, (int)tiles};
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
    default: GO(64, 64, 2, 2, 4) break;
  }
#undef GO
  HIP_CHECK_KERNEL();
  return hipSuccess;
}

// Products of 65 to 256 rows for the few-row entry points, K in parts so that the
// blocks come to one or two a compute unit. Where M is narrow a block takes 64
// features (few parts, so few sums to add); otherwise, above 128 rows, 128 features
// and all rows. us, here / the few-row kernel, with the sums added: K 4096, M 4096 at
// 128 rows 15.9 / 18.9 (level at 77, the products alone); K 8192, M 2048 at 77 / 256 15.4 / 18.4, 21.3 /
// 29.2; K 14336, M 4096 at 200 / 256 41.4 / 49.5, 45.8 / 54.7 (54.9 with 64 features); K
// 4096, M 6144 at 256 31.9 / 33.6. Up to 128 rows the few-row kernel keeps wide M and
// long K (K 14336, M 4096 at 77 rows 29.7, 128 x 128 here 34.1).
static bool mid_narrow(int M, int K) { return M <= 4096 && K <= 8192; }

// Wide products of 65 to 128 rows in one round of blocks of 64 features and all rows, 8
// waves, K in one part. Bound by the reads of W and, per unit, as many of x. us, here /
// the few-row kernel / the library at 65 and 128 rows, weights not in a cache: K 512, M
// 10304 5.6 / 11.3 / 10.0, 6.1 / 15.8 / 10.5; K 1088, M 16384 9.5 / 15.2 / 14.6, 11.2 / 19.5
// / 14.8; K 1984, M 10304 13.1 / 15.9 / 21.0, 16.0 / 20.4 / 21.7; K 2304, M 12288 15.4 / 19.2 /
// 17.6, 18.9 / 24.6 / 20.5; K 3072, M 16384 21.3 / 25.0 / 24.0, 26.6 / 30.8 / 27.2; K 4096, M
// 14336 25.3 / 28.0 / 30.5, 29.9 / 35.2 / 33.0; K 4608, M 16384 29.9 / 33.6 / 32.7, 36.6 / 40.2 /
// 36.8. Not past K 4608, where it turns (K 5120, M 12288 at 65 / 112 rows 32.1 / 33.9 / 33.3,
// 37.5 / 39.9 / 36.0, M 16384 at 128 43.9 / 44.9 / 41.5), nor where K is long and a quarter of
// the units idle (K 4096, M 10304 23.8 / 22.4 / 38.7, 28.2 / 28.4 / 30.6); past 256 tiles a
// second round is nearly empty (K 2048, M 17408 26.4 / 23.3 / 27.5). The line at 129 tiles is
// from weights that came through the caches (K 2048, M 8192 at 128 rows 16.9 / 18.8 / 15.7);
// as they are loaded now these are ahead at 128 too (14.8 / 18.2 / 15.8, K 512 6.5 / 14.3 /
// 9.9), and it could be lower.
static bool mid_wide(int M, int K, int N) {
  const int tiles = (M + 63) / 64;
  return N > 64 && N <= 128 && tiles <= UNITS && K >= 512 && K <= 4608 &&
         (K <= 2048 ? tiles > 128 : tiles >= 192);
}
extern "C" int ks_mid_wide(int M, int K, int N) { return mid_wide(M, K, N); }

extern "C" int ks_mid_takes(int M, int K, int N) {
  if (K >= 1 << 22) return 0;  // (offsets within a tile of 32 bits)
  return N > 128 || (N > (M < 4096 ? 64 : 96) && mid_narrow(M, K)) || mid_wide(M, K, N);
}

extern "C" int ks_mid_splits(int M, int K, int N) {
  if (mid_wide(M, K, N)) return 1;
  const int tm = mid_narrow(M, K) ? 64 : 128;
  const int tiles = (M + tm - 1) / tm * (tm == 64 && N > 128 ? 2 : 1);
  int s = UNITS / (tiles > 0 ? tiles : 1);
  if (s > K / BK / 4) s = K / BK / 4;
  return s < 1 ? 1 : s > 16 ? 16 : s;
}

// out: fp32 sums of the parts (sums) or bf16 with the bias, if there is one
extern "C" hipError_t ks_mid_gemm(void* out, const void* x, const void* w,
                                  const void* bias, int M, int K, int N, long xs,
                                  int splits, int sums, hipStream_t stream) {
  if ((bias && (sums || M % 8 != 0)) || N < 1 || N > 256 || M < 4 || M % 4 != 0 || K < BK || K % BK != 0 ||
      K >= 1 << 22 || xs % 8 != 0 || xs >= 1 << 22 || splits < 1 || splits > K / BK ||
      (splits > 1 && !sums) ||
      (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out | (uintptr_t)bias) & 15) != 0)
    return hipErrorInvalidValue;
  DenseArgs p{out, (const short*)x, (const short*)w, (const short*)bias, M, K, N, (int)xs,
              0, 0};
#define GO(tn, tm, wn, wm, s, epi)                                                    \
  {                                                                                   \
    p.ftiles = (M + tm - 1) / tm;                                                     \
    p.tiles = p.ftiles * ((N + tn - 1) / tn);                                         \
    hipLaunchKernelGGL((dense_gemm_kernel<tn, tm, wn, wm, s, epi>),                   \
                       dim3(p.tiles, splits), dim3(wn * wm * 64), 0, stream, p);      \
  }
  if (mid_narrow(M, K) || mid_wide(M, K, N)) {
    if (sums) GO(128, 64, 2, 2, 3, PARTIAL)
    else GO(128, 64, 4, 2, 4, BIAS)
  } else {
    if (sums) GO(256, 128, 4, 2, 3, PARTIAL)
    else GO(256, 128, 4, 2, 3, BIAS)
  }
#undef GO
  HIP_CHECK_KERNEL();
  return hipSuccess;
}
