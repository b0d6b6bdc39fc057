// Rotary position embedding (neox-style rotate-half), in-place on q and k.
//
// cos/sin table is host-precomputed (CDNA guide Appendix B: no on-device
// trig) as [max_pos, head_dim] f32 = [cos(half) | sin(half)].
#include "common.h"

namespace {

// One wave per (token, head). lane i < half handles dim pair (i, i+half).
// head_dim <= 128 assumed per wave pass (loops for larger).
__global__ void rope_kernel(short* __restrict__ q,  // [T, Hq, D] (row stride sq)
                            short* __restrict__ k,  // [T, Hk, D] (row stride sk)
                            const long* __restrict__ positions,  // [T]
                            const float* __restrict__ cos_sin,   // [P, D]
                            const int T, const int Hq, const int Hk,
                            const int D, const long sq, const long sk) {
  const int half = D >> 1;
  const int waves_per_block = blockDim.x >> 6;
  const int gwave = blockIdx.x * waves_per_block + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int total_heads = Hq + Hk;
  const long total_waves = (long)T * total_heads;
  if (gwave >= total_waves) return;
  const int t = gwave / total_heads;
  const int h = gwave % total_heads;
  const long pos = positions[t];
  const float* cs = cos_sin + pos * D;
  short* base = (h < Hq) ? q + (long)t * sq + (long)h * D
                         : k + (long)t * sk + (long)(h - Hq) * D;
  for (int i = lane; i < half; i += 64) {
    float c = cs[i];
    float s = cs[half + i];
    float x1 = bf16_bits_to_float(base[i]);
    float x2 = bf16_bits_to_float(base[i + half]);
    base[i] = float_to_bf16_bits(x1 * c - x2 * s);
    base[i + half] = float_to_bf16_bits(x2 * c + x1 * s);
  }
}

// Rotation of q and k and the scatter of k and v into the page pool in one
// pass. A lane takes eight dims of each half of a head, so a head is D / 16
// lanes and a wave several heads of one token, which share the lane's cosines
// and sines. SPLITS: q, k and v are the fp32 K-split sums of their projection,
// added here in order, and the bf16 rows are written whole (they are what
// attention over the chunk itself reads).
//
// Bound by memory for long prompts (8191 tokens of 32 + 8 + 8 heads of 128:
// 41 us = 4.9 TB/s where the two kernels took 73 + 13), by the launch for decode
// steps, where this takes 4.8 us for three of 4.7 (sum of splits, rotation,
// scatter; 1 to 77 rows).
struct RopeCacheArgs {
  short *q, *k, *v;     // [T][heads][D], row strides sq, sk, sv
  const float* part;    // SPLITS: [splits][T][(Hq + 2 Hk) D]
  int splits;
  const long* positions;
  const float* cos_sin;
  void *k_cache, *v_cache;  // [pages][Hk][block][D] or null
  const int* slots;
  int T, Hq, Hk, D, block;
  long sq, sk, sv;
};

__device__ __forceinline__ void store_page(short* p, const short8_t v) {
  *reinterpret_cast<short8_t*>(p) = v;
}
__device__ __forceinline__ void store_page(unsigned char* p, const short8_t v) {
  int lo = 0, hi = 0;
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(bf16_bits_to_float(v[0]), bf16_bits_to_float(v[1]), lo, false);
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(bf16_bits_to_float(v[2]), bf16_bits_to_float(v[3]), lo, true);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(bf16_bits_to_float(v[4]), bf16_bits_to_float(v[5]), hi, false);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(bf16_bits_to_float(v[6]), bf16_bits_to_float(v[7]), hi, true);
  *reinterpret_cast<int2*>(p) = int2{lo, hi};
}

template <bool SPLITS, typename CACHE>
__global__ __launch_bounds__(256) void rope_cache_kernel(const RopeCacheArgs p) {
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= p.T) return;
  const int per = p.D >> 4, half = p.D >> 1;  // lanes of a head
  const int hpw = 64 / per;                   // heads of a wave
  const int sub = lane / per;
  if (sub >= hpw) return;
  const int d0 = (lane - sub * per) * 8;
  const float* cs = p.cos_sin + p.positions[t] * (long)p.D + d0;
  float c[8], s[8];
#pragma unroll
  for (int e = 0; e < 8; e += 4) {
    *reinterpret_cast<float4_t*>(c + e) = *reinterpret_cast<const float4_t*>(cs + e);
    *reinterpret_cast<float4_t*>(s + e) = *reinterpret_cast<const float4_t*>(cs + half + e);
  }
  int slot = -1;
  if (p.k_cache) slot = p.slots[t];
  const int page = slot >= 0 ? slot / p.block : 0;
  const int at = slot >= 0 ? slot - page * p.block : 0;
  const int heads = p.Hq + 2 * p.Hk;
  const long row = (long)heads * p.D, nm = row * p.T;

  for (int h = blockIdx.y * hpw + sub; h < heads; h += gridDim.y * hpw) {
    const int kind = h < p.Hq ? 0 : h < p.Hq + p.Hk ? 1 : 2;
    short* base = kind == 0   ? p.q + t * p.sq + (long)h * p.D
                  : kind == 1 ? p.k + t * p.sk + (long)(h - p.Hq) * p.D
                              : p.v + t * p.sv + (long)(h - p.Hq - p.Hk) * p.D;
    base += d0;
    short8_t o1, o2;
    float x1[8], x2[8];
    if constexpr (SPLITS) {
      const float* src = p.part + t * row + (long)h * p.D + d0;
#pragma unroll
      for (int e = 0; e < 8; ++e) x1[e] = x2[e] = 0.f;
#pragma unroll 4
      for (int i = 0; i < p.splits; ++i, src += nm) {
#pragma unroll
        for (int e = 0; e < 8; e += 4) {
          const float4_t a = *reinterpret_cast<const float4_t*>(src + e);
          const float4_t b = *reinterpret_cast<const float4_t*>(src + half + e);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            x1[e + j] += a[j];
            x2[e + j] += b[j];
          }
        }
      }
    } else {
      o1 = *reinterpret_cast<const short8_t*>(base);
      o2 = *reinterpret_cast<const short8_t*>(base + half);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        x1[e] = bf16_bits_to_float(o1[e]);
        x2[e] = bf16_bits_to_float(o2[e]);
      }
    }
    if (kind < 2) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        o1[e] = float_to_bf16_bits(x1[e] * c[e] - x2[e] * s[e]);
        o2[e] = float_to_bf16_bits(x2[e] * c[e] + x1[e] * s[e]);
      }
    } else if constexpr (SPLITS) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        o1[e] = float_to_bf16_bits(x1[e]);
        o2[e] = float_to_bf16_bits(x2[e]);
      }
    }
    if (SPLITS || kind < 2) {
      *reinterpret_cast<short8_t*>(base) = o1;
      *reinterpret_cast<short8_t*>(base + half) = o2;
    }
    if (kind > 0 && slot >= 0) {
      const int hk = h - p.Hq - (kind == 2 ? p.Hk : 0);
      CACHE* to = reinterpret_cast<CACHE*>(kind == 1 ? p.k_cache : p.v_cache) +
                  (((long)page * p.Hk + hk) * p.block + at) * p.D + d0;
      store_page(to, o1);
      store_page(to + half, o2);
    }
  }
}

}  // namespace

// Rotates q and k in place (splits 0) or out of the K-split sums `part`, and
// scatters k and v into the pages unless k_cache is null.
extern "C" hipError_t ks_rope_cache(void* q, void* k, void* v, const void* part,
                                    int splits, const void* positions,
                                    const void* cos_sin, void* k_cache,
                                    void* v_cache, const void* slots, int T, int Hq,
                                    int Hk, int D, int block, int fp8, long sq,
                                    long sk, long sv, hipStream_t stream) {
  if (T == 0) return hipSuccess;
  if (T < 0 || D % 16 != 0 || D < 16 || D > 1024 || Hq + Hk < 1 ||
      (k_cache && block < 1) || (sq | sk | sv) % 8 != 0 || (splits > 0) != (part != nullptr) ||
      (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)part |
        (uintptr_t)cos_sin | (uintptr_t)k_cache | (uintptr_t)v_cache) & 15) != 0)
    return hipErrorInvalidValue;
  const RopeCacheArgs p{(short*)q, (short*)k, (short*)v, (const float*)part, splits,
                        (const long*)positions, (const float*)cos_sin, k_cache,
                        v_cache, (const int*)slots, T, Hq, Hk, D, block, sq, sk, sv};
  // heads go over more blocks until there are four per compute unit
  const int groups = (Hq + 2 * Hk + 64 / (D / 16) - 1) / (64 / (D / 16));
  const int bx = (T + 3) / 4;
  int by = (1024 + bx - 1) / bx;
  if (by > groups) by = groups;
  const dim3 grid(bx, by);
#define GO(S, C) \
  hipLaunchKernelGGL((rope_cache_kernel<S, C>), grid, dim3(256), 0, stream, p)
  if (splits > 0) {
    if (fp8) GO(true, unsigned char);
    else GO(true, short);
  } else {
    if (fp8) GO(false, unsigned char);
    else GO(false, short);
  }
#undef GO
  HIP_CHECK_KERNEL();
  return hipSuccess;
}

extern "C" hipError_t ks_rotary_embedding(void* q, void* k,
                                          const void* positions,
                                          const void* cos_sin, int T, int Hq,
                                          int Hk, int D, long sq, long sk,
                                          hipStream_t stream) {
  if (D % 2 != 0) return hipErrorInvalidValue;
  const long total_waves = (long)T * (Hq + Hk);
  if (total_waves == 0) return hipSuccess;
  const int waves_per_block = 4;  // 256 threads
  int grid = (int)((total_waves + waves_per_block - 1) / waves_per_block);
  hipLaunchKernelGGL(rope_kernel, dim3(grid), dim3(256), 0, stream, (short*)q,
                     (short*)k, (const long*)positions, (const float*)cos_sin,
                     T, Hq, Hk, D, sq, sk);
  HIP_CHECK_KERNEL();
  return hipSuccess;
}
