// State-space (Mamba-2 / SSD form) sequence mixer kernels over a flat,
// variable-length token batch with per-sequence state slots.
//
// A sequence's portion may start anywhere: `positions[t]` is the absolute
// position of token t, `seq_of_token[t]` its sequence in the batch,
// `cu_seqlens[s]` the first flat token of sequence s and `slots[s]` the row
// of the state pools that carries it between steps. A portion that starts at
// position 0 ignores whatever its slot held (slots are reused, never cleared).
//
//  * causal_conv_silu: depthwise causal convolution over `taps` inputs per
//    channel + bias (optional) + silu (optional). Inputs before the portion come from the conv
//    state (the last taps-1 raw inputs of the sequence), zeros before
//    position 0.
//  * conv_state_update: runs after the above, shifts the new raw inputs in
//    (short portions: one kernel does both).
//  * ssd_scan: per head h with group g(h):
//        a_t = exp(-exp(A_log_h) * dt_t),  dt_t = softplus(dt_raw + dt_bias_h)
//        S_t = a_t S_{t-1} + dt_t B_t x_t^T        (S: N x P, fp32)
//        y_t = S_t^T C_t + D_h x_t
//    The state lives in registers: lane (ns, pl) owns rows n = ns + 16 r of
//    a few columns of one head, a 16-lane shuffle tree sums the C-contraction.
//    Tokens of a sequence are walked in order, a chunk at a time through LDS.
//    Serves prefill portions and single-token decode alike (grid = column
//    tiles x heads x sequences, so decode batches fill the chip).
#include "dtype_io.h"

#include <float.h>
#include <type_traits>

namespace {

constexpr int MAX_TAPS = 16;

// sum over each row of 16 lanes with DPP lane swaps (VALU rate, no LDS
// traffic): swap within pairs, within quads, mirror the 8-lane half, mirror
// the row; every lane of the row ends with the row's sum
__device__ __forceinline__ float row16_sum(float v) {
  auto swz = [](float x, auto ctrl) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x),
                                           decltype(ctrl)::value, 0xF, 0xF, true));
  };
  v += swz(v, std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]
  v += swz(v, std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
  v += swz(v, std::integral_constant<int, 0x141>{});  // row_half_mirror
  v += swz(v, std::integral_constant<int, 0x140>{});  // row_mirror
  return v;
}

__device__ __forceinline__ float silu_f(float v) {
  return v / (1.0f + expf(-v));
}

template <typename T>
__global__ void causal_conv_silu_kernel(
    float* __restrict__ out, const T* __restrict__ in, long in_stride,
    const float* __restrict__ w, const float* __restrict__ bias,
    const T* __restrict__ conv_state, const long* __restrict__ positions,
    const int* __restrict__ seq_of_token, const int* __restrict__ cu_seqlens,
    const int* __restrict__ slots, int channels, int taps, int silu) {
  const int t = blockIdx.y;
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= channels) return;
  const int s = seq_of_token[t];
  const int first = cu_seqlens[s];
  const long pos = positions[t];
  const long slot = slots[s];
  const int hist = taps - 1;
  float acc = bias ? bias[c] : 0.f;
  for (int j = 0; j < taps; ++j) {
    const int back = hist - j;  // 0 = the current token
    if (pos - back < 0) continue;
    float v;
    if (t - back >= first) {
      v = ld_f32(in, (long)(t - back) * in_stride + c);
    } else {
      // state row i holds the input at position (portion start - hist + i)
      const int i = hist - back + (t - first);
      v = ld_f32(conv_state, (slot * hist + i) * channels + c);
    }
    acc += w[(long)c * taps + j] * v;
  }
  out[(long)t * channels + c] = silu ? silu_f(acc) : acc;
}

// 4 consecutive channels per lane (8- or 16-byte loads, 16-byte stores); the
// launcher picks it when pointers, strides and the channel count allow
template <typename T>
__device__ __forceinline__ void load4(const T* p, float* v);
template <>
__device__ __forceinline__ void load4<short>(const short* p, float* v) {
  const short4_t x = *reinterpret_cast<const short4_t*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = bf16_bits_to_float(x[i]);
}
template <>
__device__ __forceinline__ void load4<float>(const float* p, float* v) {
  const float4_t x = *reinterpret_cast<const float4_t*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = x[i];
}

// A block of the vector kernel takes 4 tokens, or 16 where inputs and outputs
// are more than the memory-side cache holds (256 MB: 6 bytes an element with
// bf16 in). The last TAPS - 1 inputs stay in registers while a lane walks its
// tokens, so a token costs one load and a block TAPS - 1 more; these come from a
// cache up to there, while the loads of a walk are one after the other and short
// portions start it anew (with the state update, us, 4 / 16 tokens, 6144
// channels: 500 tokens 11 / 16, 6000 48 / 48, 8000 75 / 70; 127 sequences of 1
// and one of 385 23 / 39; 10240 channels, 6000 tokens 103 / 85). Bound by memory and
// the exact exponential: 8000 tokens of 6144 channels 55 us = 5.3 TB/s without the
// update (59.5 with one load under way at a time).
constexpr int CONV_TT = 4, CONV_TT_LONG = 16;
constexpr long CONV_LONG = 42L << 20;  // tokens x channels

template <typename T, int TAPS, int TT>
__global__ __launch_bounds__(256) void causal_conv_silu_vec4_kernel(
    float* __restrict__ out, const T* __restrict__ in, long in_stride,
    const float* __restrict__ w, const float* __restrict__ bias,
    const T* __restrict__ conv_state, const long* __restrict__ positions,
    const int* __restrict__ seq_of_token, const int* __restrict__ cu_seqlens,
    const int* __restrict__ slots, int tokens, int channels, int silu) {
  const int c = (blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (c >= channels) return;
  constexpr int hist = TAPS - 1;
  // taps and bias of this lane's 4 channels, reused for every token
  float wt[4][TAPS], b4[4];
  if (bias) load4<float>(bias + c, b4);
  else b4[0] = b4[1] = b4[2] = b4[3] = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < TAPS; ++j) wt[i][j] = w[(long)(c + i) * TAPS + j];
  const int t0 = blockIdx.y * TT;
  const int t_end = min(tokens, t0 + TT);
  float win[TAPS][4];  // inputs of tokens t - hist .. t
  int end = 0;         // first token after the sequence that t is in
  float ahead[4][4];   // four tokens' loads are under way at a time
#pragma unroll 1
  for (int t4 = t0; t4 < t_end; t4 += 4) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      load4<T>(in + (long)min(t4 + u, t_end - 1) * in_stride + c, ahead[u]);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = t4 + u;
      if (t >= t_end) break;
      if (t == t0 || t >= end) {  // the inputs before t, from the rows or the state
        const int s = seq_of_token[t];
        const int first = cu_seqlens[s];
        end = cu_seqlens[s + 1];
        const long pos = positions[t];
        const long slot = slots[s];
#pragma unroll
        for (int back = hist; back > 0; --back) {
          float* v = win[hist - back];
          if (pos - back < 0)
            v[0] = v[1] = v[2] = v[3] = 0.f;
          else if (t - back >= first)
            load4<T>(in + (long)(t - back) * in_stride + c, v);
          else
            load4<T>(conv_state + (slot * hist + (hist - back + (t - first))) * channels + c,
                     v);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) win[hist][i] = ahead[u][i];
      float acc[4] = {b4[0], b4[1], b4[2], b4[3]};
#pragma unroll
      for (int j = 0; j < TAPS; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] += wt[i][j] * win[j][i];
      float4_t o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = silu ? silu_f(acc[i]) : acc[i];
      *reinterpret_cast<float4_t*>(out + (long)t * channels + c) = o;
#pragma unroll
      for (int j = 0; j < hist; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) win[j][i] = win[j + 1][i];
    }
  }
}

// A block walks the whole portion of one sequence and leaves its conv state:
// one launch where the portions are short (decode steps), with the state read
// once. 128 sequences of one token, 6144 channels: 7.6 us, 21 for the kernel
// above and the state update.
template <typename T, int TAPS>
__global__ __launch_bounds__(256) void causal_conv_silu_seq_kernel(
    float* __restrict__ out, const T* __restrict__ in, long in_stride,
    const float* __restrict__ w, const float* __restrict__ bias,
    T* __restrict__ conv_state, const long* __restrict__ positions,
    const int* __restrict__ cu_seqlens, const int* __restrict__ slots,
    int channels, int silu) {
  const int c = (blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (c >= channels) return;
  constexpr int hist = TAPS - 1;
  typedef T vec4 __attribute__((ext_vector_type(4)));
  const int s = blockIdx.y;
  const int first = cu_seqlens[s], end = cu_seqlens[s + 1];
  if (end <= first) return;
  const long start = positions[first];
  vec4* st = reinterpret_cast<vec4*>(conv_state + (long)slots[s] * hist * channels + c);
  const int row = channels / 4;
  vec4 raw[TAPS];
#pragma unroll
  for (int i = 0; i < hist; ++i)
    raw[i] = start - hist + i < 0 ? vec4{0, 0, 0, 0} : st[(long)i * row];
  float wt[4][TAPS], b4[4];
  if (bias) load4<float>(bias + c, b4);
  else b4[0] = b4[1] = b4[2] = b4[3] = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < TAPS; ++j) wt[i][j] = w[(long)(c + i) * TAPS + j];
  for (int t = first; t < end; ++t) {
    raw[hist] = *reinterpret_cast<const vec4*>(in + (long)t * in_stride + c);
    float4_t o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float acc = b4[i];
#pragma unroll
      for (int j = 0; j < TAPS; ++j) {
        const T v = raw[j][i];
        acc += wt[i][j] * ld_f32(&v, 0);
      }
      o[i] = silu ? silu_f(acc) : acc;
    }
    *reinterpret_cast<float4_t*>(out + (long)t * channels + c) = o;
#pragma unroll
    for (int j = 0; j < hist; ++j) raw[j] = raw[j + 1];
  }
#pragma unroll
  for (int i = 0; i < hist; ++i) st[(long)i * row] = raw[i];
}

template <typename T>
__global__ void conv_state_update_kernel(
    T* __restrict__ conv_state, const T* __restrict__ in, long in_stride,
    const long* __restrict__ positions, const int* __restrict__ cu_seqlens,
    const int* __restrict__ slots, int channels, int taps) {
  const int s = blockIdx.y;
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= channels) return;
  const int first = cu_seqlens[s];
  const int len = cu_seqlens[s + 1] - first;
  if (len <= 0) return;
  const long start = positions[first];
  const long slot = slots[s];
  const int hist = taps - 1;
  T keep[MAX_TAPS];
  // new row i holds position (start + len - hist + i)
  for (int i = 0; i < hist; ++i) {
    const long rel = (long)len - hist + i;  // offset into the portion
    T v;
    if (rel >= 0) {
      v = in[(first + rel) * in_stride + c];
    } else if (start + rel < 0) {
      st_f32(&v, 0, 0.f);
    } else {
      v = conv_state[(slot * hist + (hist + rel)) * channels + c];
    }
    keep[i] = v;
  }
  for (int i = 0; i < hist; ++i)
    conv_state[(slot * hist + i) * channels + c] = keep[i];
}

// R = state rows per lane (N <= 16 R), PC = columns per lane (tile of 16 PC
// columns of one head per block). blockDim = 256 = 16 row-lanes x 16 col-lanes.
// Tokens are taken in chunks of `tc`: the chunk's B, C, x rows and step sizes
// are staged in LDS with coalesced loads (the next chunk's loads are in
// flight while this one is computed), softplus/exp run once per (token, head)
// instead of once per lane, and y leaves through LDS as whole rows.
constexpr int SCAN_TC = 16;  // tokens per chunk

template <int R, int PC>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
ssd_scan_kernel(
    float* __restrict__ y, const float* __restrict__ xbc,
    const float* __restrict__ dt_raw_f32, const short* __restrict__ dt_raw_bf16,
    long dt_stride, const float* __restrict__ dt_bias,
    const float* __restrict__ a_log, const float* __restrict__ d_skip,
    float* __restrict__ state, const long* __restrict__ positions,
    const int* __restrict__ cu_seqlens, const int* __restrict__ slots,
    int heads, int groups, int P, int N) {
  extern __shared__ float lds[];
  constexpr int tc = SCAN_TC;
  const int s = blockIdx.z;
  const int h = blockIdx.y;
  const int ns = threadIdx.x & 15;
  const int pl = threadIdx.x >> 4;
  const int p0 = blockIdx.x * (16 * PC);
  const int pt = min(16 * PC, P - p0);  // columns of this tile
  const int first = cu_seqlens[s];
  const int len = cu_seqlens[s + 1] - first;
  if (len <= 0) return;
  const int g = h / (heads / groups);
  const int inner = heads * P;
  const int channels = inner + 2 * groups * N;
  const long slot = slots[s];
  const bool fresh = positions[first] == 0;
  const float A = -expf(a_log[h]);
  const float bias = dt_bias[h];
  const float Dh = d_skip[h];

  // LDS: B[tc][N] | C[tc][N] | x[tc][16 PC] | dt[tc] | decay[tc] | y[tc][16 PC]
  const int XS = 16 * PC;
  float* Bs = lds;
  float* Cs = Bs + tc * N;
  float* Xs = Cs + tc * N;
  float* Ds = Xs + tc * XS;
  float* As = Ds + tc;
  float* Ys = As + tc;
  float S[R][PC];
  float* sp = state + ((slot * heads + h) * (long)P) * N;
#pragma unroll
  for (int c = 0; c < PC; ++c) {
    const int p = p0 + pl + 16 * c;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int n = ns + 16 * r;
      S[r][c] = (!fresh && p < P && n < N) ? sp[(long)p * N + n] : 0.f;
    }
  }

  // staging: 16 threads per token of the chunk, each takes every 16th
  // element of the token's B, C and x rows (no index arithmetic beyond adds)
  const int stk = threadIdx.x >> 4;   // token of the chunk this thread stages
  const int sl = threadIdx.x & 15;
  float sB[R], sC[R], sX[PC], sdt = 0.f;
  auto prefetch = [&](int t0, int cnt) {
    if (stk < cnt) {
      const long t = first + t0 + stk;
      const float* row = xbc + t * channels;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int n = sl + 16 * r;
        sB[r] = n < N ? row[inner + g * N + n] : 0.f;
        sC[r] = n < N ? row[inner + groups * N + g * N + n] : 0.f;
      }
#pragma unroll
      for (int c = 0; c < PC; ++c) {
        const int col = sl + 16 * c;
        sX[c] = col < pt ? row[h * P + p0 + col] : 0.f;
      }
      if (sl == 0) {
        const long i = t * dt_stride + h;
        sdt = (dt_raw_f32 ? dt_raw_f32[i] : bf16_bits_to_float(dt_raw_bf16[i])) + bias;
      }
    }
  };
  auto commit = [&](int cnt) {
    if (stk < cnt) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int n = sl + 16 * r;
        if (n < N) {
          Bs[stk * N + n] = sB[r];
          Cs[stk * N + n] = sC[r];
        }
      }
#pragma unroll
      for (int c = 0; c < PC; ++c) Xs[stk * XS + sl + 16 * c] = sX[c];
      if (sl == 0) {
        // softplus without a clamp; log1p(exp(v)) is v itself past v ~ 30
        const float dt = sdt > 30.f ? sdt : log1pf(expf(sdt));
        Ds[stk] = dt;
        As[stk] = expf(A * dt);
      }
    }
  };

  prefetch(0, min(tc, len));
  for (int t0 = 0; t0 < len; t0 += tc) {
    const int cnt = min(tc, len - t0);
    __syncthreads();  // previous chunk's LDS fully consumed
    commit(cnt);
    __syncthreads();
    if (t0 + tc < len) prefetch(t0 + tc, min(tc, len - t0 - tc));
    for (int tk = 0; tk < cnt; ++tk) {
      const float a = As[tk], dt = Ds[tk];
      float B[R], C[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int n = ns + 16 * r;
        const bool ok = n < N;
        B[r] = ok ? Bs[tk * N + n] : 0.f;
        C[r] = ok ? Cs[tk * N + n] : 0.f;
      }
#pragma unroll
      for (int c = 0; c < PC; ++c) {
        const int col = pl + 16 * c;
        const float x = col < pt ? Xs[tk * XS + col] : 0.f;
        const float dtx = dt * x;
        float acc = 0.f;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          S[r][c] = a * S[r][c] + B[r] * dtx;
          acc += S[r][c] * C[r];
        }
        acc = row16_sum(acc);
        if (ns == 0) Ys[tk * XS + col] = acc + Dh * x;
      }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < cnt * pt; e += 256) {
      const int tk = e / pt, col = e % pt;
      y[(long)(first + t0 + tk) * inner + h * P + p0 + col] = Ys[tk * XS + col];
    }
  }
#pragma unroll
  for (int c = 0; c < PC; ++c) {
    const int p = p0 + pl + 16 * c;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int n = ns + 16 * r;
      if (p < P && n < N) sp[(long)p * N + n] = S[r][c];
    }
  }
}

// sums of V[0 .. NP) over groups of NL lanes, each level handing half of the
// values that are left to the other half of the lanes: lane nl of a group ends
// with the sum of V[nl / 4] (NP = NL / 4 values)
template <int NL, int NP>
__device__ __forceinline__ float group_sums(float (&V)[NP], const int nl) {
  static_assert(NP == NL / 4 && (NL == 16 || NL == 32), "lanes");
  auto dpp = [](float x, auto ctrl) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x),
                                           decltype(ctrl)::value, 0xF, 0xF, true));
  };
  if constexpr (NL == 32) {  // rows of 16 lanes: odd ones take V[4 ..]
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const auto r = __builtin_amdgcn_permlane16_swap(
          __builtin_bit_cast(unsigned int, V[i]),
          __builtin_bit_cast(unsigned int, V[i + 4]), false, false);
      V[i] = __builtin_bit_cast(float, (unsigned int)r[0]) +
             __builtin_bit_cast(float, (unsigned int)r[1]);
    }
  }
  const bool half = nl & 8, quad = nl & 4;
#pragma unroll
  for (int i = 0; i < 2; ++i)  // halves of a row, mirrored
    V[i] = (half ? V[i + 2] : V[i]) +
           dpp(half ? V[i] : V[i + 2], std::integral_constant<int, 0x140>{});
  float v = (quad ? V[1] : V[0]) +  // quads of a half row, mirrored
            dpp(quad ? V[0] : V[1], std::integral_constant<int, 0x141>{});
  v += dpp(v, std::integral_constant<int, 0xB1>{});
  v += dpp(v, std::integral_constant<int, 0x4E>{});
  return v;
}

// The scan for portions of a token or two (decode steps), bound by the state's
// way through memory: NL lanes hold a state row, 16 bytes each, so a wave reads
// and writes whole rows, and a block's 64 columns of one head are all in flight
// before the first token is there. What the vector units do beside it has to
// stay below that: uniform addresses, sums that halve their values as they go
// (with whole butterflies 770 us where this takes 401). 512 sequences of one
// token, 64 heads of 64 x 128: 401 us = 5.4 TB/s, 594 us with the kernel above;
// 128 sequences 83 and 153 us.
template <int NL>  // lanes of a state row: N = 4 NL
__global__ void __launch_bounds__(256) ssd_step_kernel(
    float* __restrict__ y, const float* __restrict__ xbc,
    const float* __restrict__ dt_raw_f32, const short* __restrict__ dt_raw_bf16,
    long dt_stride, const float* __restrict__ dt_bias,
    const float* __restrict__ a_log, const float* __restrict__ d_skip,
    float* __restrict__ state, const long* __restrict__ positions,
    const int* __restrict__ cu_seqlens, const int* __restrict__ slots,
    int heads, int groups, int P) {
  constexpr int N = 4 * NL;
  constexpr int RP = 256 / NL;   // state rows (columns p) per pass
  constexpr int NP = 64 / RP;    // passes
  const int s = blockIdx.z, h = blockIdx.y, p0 = blockIdx.x * 64;
  const int first = cu_seqlens[s], end = cu_seqlens[s + 1];
  if (end <= first) return;
  const unsigned nl = threadIdx.x % NL, pl = threadIdx.x / NL, n = nl * 4;
  const bool fresh = positions[first] == 0;
  float* sp = state + (((long)slots[s] * heads + h) * P + p0) * N;
  const unsigned at = pl * N + n;
  float4_t S[NP];
  if (fresh) {
#pragma unroll
    for (int i = 0; i < NP; ++i) S[i] = float4_t{0.f, 0.f, 0.f, 0.f};
  } else {
#pragma unroll
    for (int i = 0; i < NP; ++i)
      S[i] = __builtin_nontemporal_load(
          reinterpret_cast<const float4_t*>(sp + RP * i * N + at));
  }
  const int g = h / (heads / groups), inner = heads * P;
  const long channels = inner + 2L * groups * N;
  const float A = -expf(a_log[h]), bias = dt_bias[h], Dh = d_skip[h];
  for (int t = first; t < end; ++t) {
    const float* row = xbc + t * channels;
    const float* xr = row + h * P + p0;
    const float* br = row + inner + g * N;
    const float4_t B = *reinterpret_cast<const float4_t*>(br + n);
    const float4_t C = *reinterpret_cast<const float4_t*>(br + groups * N + n);
    float x[NP], acc[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) x[i] = xr[RP * i + pl];
    const long di = t * dt_stride + h;
    const float v = (dt_raw_f32 ? dt_raw_f32[di] : bf16_bits_to_float(dt_raw_bf16[di])) + bias;
    // softplus without a clamp; log1p(exp(v)) is v itself past v ~ 30
    const float dt = v > 30.f ? v : log1pf(expf(v));
    const float a = expf(A * dt);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const float dtx = dt * x[i];
      acc[i] = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        S[i][j] = fmaf(a, S[i][j], B[j] * dtx);
        acc[i] += S[i][j] * C[j];
      }
    }
    const float sum = group_sums<NL, NP>(acc, nl);
    const int i = nl / 4;  // the pass whose row this lane has the sum of
    if (nl % 4 == 0)
      y[(long)t * inner + h * P + p0 + RP * i + pl] = sum + Dh * xr[RP * i + pl];
  }
  // Past the caches like the loads: written back by and by, the states took the memory
  // from the products that follow (hybrid step of 1 / 72 / 128 sequences 328 -> 318, 677
  // -> 651, 975 -> 931 us).
#pragma unroll
  for (int i = 0; i < NP; ++i)
    __builtin_nontemporal_store(S[i], reinterpret_cast<float4_t*>(sp + RP * i * N + at));
}

// ---------------------------------------------------------------------------
// The scan in chunks of 64 tokens on the fp32 matrix cores
// (v_mfma_f32_16x16x4_f32), in one launch: for portions of one or two chunks (the
// form after it takes the longer ones). With c_t the running sum of A dt inside the chunk and S the state at its
// start:
//     y_t = exp(c_t) S^T C_t + sum_{s <= t} (C_t . B_s) exp(c_t - c_s) dt_s x_s
//           + D x_t
//     S  <- exp(c_end) S + sum_s exp(c_end - c_s) dt_s B_s x_s^T
// A block takes 64 columns (p) of one head of one sequence; each of its 8 waves
// owns 16 columns and half of the states, S^T in accumulator layout (row
// n = 16 nb + 4 g + r in register r of lane group g), which is already the B
// operand of C S for the contraction order "lane group g, product r -> state
// 4 g + r"; C is then read from LDS four states at a time. The waves share the
// 64 x 64 products C B^T (the 10 16 x 16 tiles on and below the diagonal); the
// two halves of a column block add their sums over states through LDS, each
// finishing half of the token tiles. The next chunk's rows are on their way in
// registers meanwhile.
//
// Bound by the products of one chunk after the other: 212 per wave of 32
// cycles each, two waves per SIMD (5.6 us of the 10 us that a chunk takes).
// Token by token a chunk took 64 times the latency of one step (LDS reads,
// update, lane tree), whatever the arithmetic. 64 heads of 64 columns, 128
// states: 1 x 40 tokens 43 -> 13 us, 4 x 64 16, 8 x 20 25.
// ---------------------------------------------------------------------------
constexpr int CQ = 64;  // tokens per chunk
constexpr int CT = 512;
typedef float f32x4s __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4s mfma4(float a, float b, f32x4s c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <int NB>  // blocks of 16 states: N <= 16 NB
__global__ void __launch_bounds__(CT) ssd_chunk_kernel(
    float* __restrict__ y, const float* __restrict__ xbc,
    const float* __restrict__ dt_raw_f32, const short* __restrict__ dt_raw_bf16,
    long dt_stride, const float* __restrict__ dt_bias,
    const float* __restrict__ a_log, const float* __restrict__ d_skip,
    float* __restrict__ state, const long* __restrict__ positions,
    const int* __restrict__ cu_seqlens, const int* __restrict__ slots,
    int heads, int groups, int P, int N) {
  constexpr int NP = NB * 16;
  constexpr int RS = NP + 4;  // B and C rows: 4 rows apart fall 16 banks apart
  constexpr int XS = 64 + 4;
  constexpr int NH = NB / 2;  // of them, a wave's own
  constexpr int NV = CQ * NP / 4 / CT;  // float4 per thread of a B or C tile
  constexpr int XV = CQ * 64 / 4 / CT;
  __shared__ __attribute__((aligned(16))) float Bs[CQ * RS];
  __shared__ __attribute__((aligned(16))) float Cs[CQ * RS];
  __shared__ __attribute__((aligned(16))) float Xs[CQ * XS];
  __shared__ __attribute__((aligned(16))) float Ms[CQ * XS];
  __shared__ __attribute__((aligned(16))) f32x4s part[CT / 64][2][64];
  __shared__ __attribute__((aligned(16))) float dts[CQ], grow[CQ], left[CQ];
  // running sums in 64 bits: their differences are exponents, and a sum over a
  // chunk may be far larger than the difference of two neighbours
  __shared__ double cum[CQ];

  const int s = blockIdx.z, h = blockIdx.y;
  const int first = cu_seqlens[s];
  const int len = cu_seqlens[s + 1] - first;
  if (len <= 0) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, g = lane >> 4;
  const int p0 = blockIdx.x * 64;
  const int pw = wave & 3, nh = wave >> 2;
  const int p = p0 + pw * 16 + col;
  const int grp = h / (heads / groups);
  const int inner = heads * P;
  const int channels = inner + 2 * groups * N;
  // finite where exp leaves the range: differences of infinite running sums
  // would be NaN where the decay is 0
  float A = -expf(a_log[h]);
  if (A < -FLT_MAX) A = -FLT_MAX;
  const float bias = dt_bias[h];
  const float Dh = d_skip[h];
  const bool fresh = positions[first] == 0;
  float* sp = state + ((slots[s] * (long)heads + h) * P + p) * N;

  f32x4s S[NH];
#pragma unroll
  for (int b = 0; b < NH; ++b) {
    const int n = (nh * NH + b) * 16 + g * 4;
    S[b] = (!fresh && p < P && n < N) ? *reinterpret_cast<const f32x4s*>(sp + n)
                                      : f32x4s{0.f, 0.f, 0.f, 0.f};
  }

  f32x4s rB[NV], rC[NV], rX[XV];
  float rdt = 0.f;
  auto fetch = [&](int t0) {
    const f32x4s zero = f32x4s{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int e = threadIdx.x + i * CT;
      const int tk = e / (NP / 4), n = e % (NP / 4) * 4;
      const bool ok = t0 + tk < len && n < N;
      const float* row = xbc + (long)(first + t0 + tk) * channels + inner + grp * N + n;
      rB[i] = ok ? *reinterpret_cast<const f32x4s*>(row) : zero;
      rC[i] = ok ? *reinterpret_cast<const f32x4s*>(row + groups * N) : zero;
    }
#pragma unroll
    for (int i = 0; i < XV; ++i) {
      const int e = threadIdx.x + i * CT;
      const int tk = e / 16, c = e % 16 * 4;
      const bool ok = t0 + tk < len && p0 + c < P;
      rX[i] = ok ? *reinterpret_cast<const f32x4s*>(
                       xbc + (long)(first + t0 + tk) * channels + h * P + p0 + c)
                 : zero;
    }
    if (wave == 0) {
      const long i = (long)(first + min(t0 + lane, len - 1)) * dt_stride + h;
      rdt = (dt_raw_f32 ? dt_raw_f32[i] : bf16_bits_to_float(dt_raw_bf16[i])) + bias;
    }
  };
  auto commit = [&](int cnt) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int e = threadIdx.x + i * CT;
      const int at = e / (NP / 4) * RS + e % (NP / 4) * 4;
      *reinterpret_cast<f32x4s*>(Bs + at) = rB[i];
      *reinterpret_cast<f32x4s*>(Cs + at) = rC[i];
    }
#pragma unroll
    for (int i = 0; i < XV; ++i) {
      const int e = threadIdx.x + i * CT;
      *reinterpret_cast<f32x4s*>(Xs + e / 16 * XS + e % 16 * 4) = rX[i];
    }
    if (wave == 0) {
      // softplus without a clamp; log1p(exp(v)) is v itself past v ~ 30.
      // Rows past the portion: dt 0, so they change nothing
      const float dt = lane < cnt ? (rdt > 30.f ? rdt : log1pf(expf(rdt))) : 0.f;
      double c = (double)A * dt;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const double o = __shfl_up(c, off, 64);
        if (lane >= off) c += o;
      }
      const double end = __shfl(c, 63, 64);
      cum[lane] = c;
      dts[lane] = dt;
      grow[lane] = expf((float)c);
      left[lane] = dt * expf((float)(end - c));
    }
  };

  fetch(0);
  for (int t0 = 0; t0 < len; t0 += CQ) {
    const int cnt = min(CQ, len - t0);
    __syncthreads();  // the previous chunk's tiles are consumed
    commit(cnt);
    __syncthreads();
    if (t0 + CQ < len) fetch(t0 + CQ);

    // ---- C B^T on and below the diagonal, with decays and step sizes ----
    for (int i = wave; i < 10; i += CT / 64) {
      const int tb = i < 1 ? 0 : i < 3 ? 1 : i < 6 ? 2 : 3;
      const int sb = i - tb * (tb + 1) / 2;
      // eight chains: fewer roundings in a row than one sum over the states
      f32x4s acc[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) acc[r] = f32x4s{0.f, 0.f, 0.f, 0.f};
      const float* ca = Cs + (tb * 16 + col) * RS + g * 4;
      const float* ba = Bs + (sb * 16 + col) * RS + g * 4;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const f32x4s c4 = *reinterpret_cast<const f32x4s*>(ca + b * 16);
        const f32x4s b4 = *reinterpret_cast<const f32x4s*>(ba + b * 16);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          f32x4s& to = acc[r + (b & 1) * 4];
          to = mfma4(c4[r], b4[r], to);
        }
      }
      const f32x4s cb = ((acc[0] + acc[1]) + (acc[2] + acc[3])) +
                        ((acc[4] + acc[5]) + (acc[6] + acc[7]));
      const int sk = sb * 16 + col;
      const double cs = cum[sk];
      const float ds = dts[sk];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int tk = tb * 16 + g * 4 + r;
        Ms[tk * XS + sk] = sk <= tk ? cb[r] * expf((float)(cum[tk] - cs)) * ds : 0.f;
      }
    }

    // ---- what the state at the chunk's start contributes ----
    f32x4s Y[4], Y2[4];
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) Y[tb] = Y2[tb] = f32x4s{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < NH; ++b) {
      f32x4s c4[4];
#pragma unroll
      for (int tb = 0; tb < 4; ++tb)
        c4[tb] = *reinterpret_cast<const f32x4s*>(Cs + (tb * 16 + col) * RS +
                                                  (nh * NH + b) * 16 + g * 4);
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int tb = 0; tb < 4; ++tb) {
          f32x4s& to = r & 1 ? Y2[tb] : Y[tb];
          to = mfma4(c4[tb][r], S[b][r], to);
        }
    }
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) Y[tb] += Y2[tb];
    // token tiles 0 and 3 are finished by the first half, 1 and 2 by the other
    part[wave][0][lane] = nh ? Y[0] : Y[1];
    part[wave][1][lane] = nh ? Y[3] : Y[2];

    // ---- the state moves on ----
    f32x4s X[4];  // token 16 tb + 4 g + r, this lane's column
#pragma unroll
    for (int tb = 0; tb < 4; ++tb)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        X[tb][r] = Xs[(tb * 16 + g * 4 + r) * XS + pw * 16 + col];
    const float keep = grow[CQ - 1];
#pragma unroll
    for (int b = 0; b < NH; ++b) S[b] *= keep;
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
      const f32x4s xw =
          X[tb] * *reinterpret_cast<const f32x4s*>(left + tb * 16 + g * 4);
      const float* brow = Bs + (tb * 16 + g * 4) * RS + nh * NH * 16 + col;
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int b = 0; b < NH; ++b)
          S[b] = mfma4(brow[r * RS + b * 16], xw[r], S[b]);
    }

    __syncthreads();  // Ms and the partial sums are complete
    // ---- what the chunk's own tokens contribute ----
    auto finish = [&](auto tile, f32x4s own, int k) {
      constexpr int tb = decltype(tile)::value;
      f32x4s acc[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] = f32x4s{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int sb = 0; sb <= tb; ++sb) {
        const f32x4s m4 = *reinterpret_cast<const f32x4s*>(
            Ms + (tb * 16 + col) * XS + sb * 16 + g * 4);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = mfma4(m4[r], X[sb][r], acc[r]);
      }
      f32x4s z = (acc[0] + acc[1]) + (acc[2] + acc[3]);
      const f32x4s e4 = *reinterpret_cast<const f32x4s*>(grow + tb * 16 + g * 4);
      const f32x4s past = (own + part[wave ^ 4][k][lane]) * e4;
      z += past;
      // The products above take later tokens of the tile with weight 0, which
      // is no 0 if their x is infinite or NaN: such sums are formed again, from
      // the tokens up to each row's own only.
      const float size = fabsf(z[0]) + fabsf(z[1]) + fabsf(z[2]) + fabsf(z[3]);
      if (__any(!(size < INFINITY))) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int tk = tb * 16 + g * 4 + r;
          float sum = 0.f;
          for (int sk = 0; sk <= tk; ++sk)
            sum = fmaf(Ms[tk * XS + sk], Xs[sk * XS + pw * 16 + col], sum);
          z[r] = sum + past[r];
        }
      }
      if (p < P) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int tk = tb * 16 + g * 4 + r;
          if (tk < cnt)
            y[(long)(first + t0 + tk) * inner + h * P + p] = z[r] + Dh * X[tb][r];
        }
      }
    };
    if (nh == 0) {
      finish(std::integral_constant<int, 0>{}, Y[0], 0);
      finish(std::integral_constant<int, 3>{}, Y[3], 1);
    } else {
      finish(std::integral_constant<int, 1>{}, Y[1], 0);
      finish(std::integral_constant<int, 2>{}, Y[2], 1);
    }
  }
#pragma unroll
  for (int b = 0; b < NH; ++b) {
    const int n = (nh * NH + b) * 16 + g * 4;
    if (p < P && n < N) *reinterpret_cast<f32x4s*>(sp + n) = S[b];
  }
}

// ---------------------------------------------------------------------------
// The same in two launches, for longer portions. What needs no state comes first,
// for all chunks at once: the products C_t . B_s of a group of heads (the 10 16 x 16
// tiles on and below the diagonal) and, per head, the running sums, these products
// with decay and step size, and the weights of the recurrence. The scan is then a
// chain of three products a chunk. A block takes 16 CB columns (p) of one head of
// one sequence. Each of its 4 waves owns a quarter of the states, S^T in
// accumulator layout, and a quarter of a chunk's tokens: it moves its states on with
// B and x from LDS, hands them to the others through LDS and forms its own tokens'
// y with C and the decayed products from registers. Two barriers a chunk; the next
// chunk's rows are on their way in registers meanwhile.
//
// The one-launch form took 10 us a chunk, 5.6 of them products: an inclusive sum in
// 64 bits, 64 x 64 exponentials and three barriers stood between them, with one
// block a compute unit. Here two blocks of 32 columns share a unit (7.8 us a chunk
// of both, 4.2 of them products, 160 per wave and block) and a block alone takes
// 4.7 us, of 16 columns 3.0. The first launch moves 19 KB a chunk and head at 4.0
// TB/s (38 us for 8000 tokens of 64 heads). us, one launch / two (64 heads of 64
// columns, 128 states): 4 x 2000 tokens 310 / 257, 1 x 2000 291 / 106, 1 x 8000
// 1156 / 390, 8 x 2000 630 / 521, 32 x 128 188 / 162, 1 x 100 21.8 / 18.0, 4 x 64
// 15.4 / 25.7. Error of y against 64 bits 8.5e-8 both.
// ---------------------------------------------------------------------------
constexpr int CTILES = 10;

// Chunks are numbered over the batch with gaps: those of sequence s from here on.
__device__ __forceinline__ int chunk_base(int first, int s) { return first / CQ + s; }

// 16 bytes at a byte offset from a uniform address, 0 past `bytes`: rows after a
// portion and columns after a head cost no branch and no address registers
__device__ __forceinline__ f32x4s load_or_zero(const float* base, unsigned int bytes,
                                               unsigned int at) {
  const __amdgpu_buffer_rsrc_t rows =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, bytes, 0x00027000);
  return __builtin_bit_cast(f32x4s, __builtin_amdgcn_raw_buffer_load_b128(rows, at, 0, 0));
}
__device__ __forceinline__ void store_or_drop(float* base, unsigned int bytes,
                                              unsigned int at, float v) {
  const __amdgpu_buffer_rsrc_t rows =
      __builtin_amdgcn_make_buffer_rsrc(base, 0, bytes, 0x00027000);
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned int, v), rows, at, 0, 0);
}
constexpr unsigned int OUTSIDE = 0x80000000u;

// tile i of the 64 x 64 products: token block tb, and the block sb <= tb before it
__device__ __forceinline__ void chunk_tile(int i, int& tb, int& sb) {
  tb = i < 1 ? 0 : i < 3 ? 1 : i < 6 ? 2 : 3;
  sb = i - tb * (tb + 1) / 2;
}

// what the scan takes per chunk and head from the pass before it
struct ChunkWork {
  f32x4s m[CTILES][64];  // tile (tb, sb) at tb (tb + 1) / 2 + sb: lane 16 g + t has
                         // (C_t . B_s) exp(c_t - c_s) dt_s for s = 4 g .. 4 g + 3
  float grow[CQ];        // exp(c_t)
  float left[CQ];        // exp(c_end - c_t) dt_t
};
constexpr int ST = 256, DT = 512, HEADS_PER_BLOCK = DT / 64;

template <int NB>  // blocks of 16 states: N <= 16 NB
__global__ void __launch_bounds__(DT) ssd_decays_kernel(
    ChunkWork* __restrict__ work, int* __restrict__ order, const float* __restrict__ xbc,
    const float* __restrict__ dt_raw_f32, const short* __restrict__ dt_raw_bf16,
    long dt_stride, const float* __restrict__ dt_bias, const float* __restrict__ a_log,
    const int* __restrict__ cu_seqlens, int seqs, int heads, int groups, int P, int N) {
  constexpr int NW = DT / 64;
  constexpr int NG = (CTILES + NW - 1) / NW;
  // running sums in 64 bits, for powers of two: their differences are exponents, and
  // a sum over a chunk may be far larger than the difference of two neighbours
  __shared__ double cum[NW][CQ];
  __shared__ float dts[NW][CQ];
  constexpr int NP = NB * 16;
  constexpr int RS = NP + 4;  // 4 rows apart fall 16 banks apart
  __shared__ __attribute__((aligned(16))) float Bs[CQ * RS];
  __shared__ __attribute__((aligned(16))) float Cs[CQ * RS];
  const int chunk = blockIdx.x;
  const int lane = threadIdx.x & 63;
  if (order && chunk == 0 && blockIdx.y == 0 && threadIdx.x < 64) {
    const int own = lane < seqs ? cu_seqlens[lane + 1] - cu_seqlens[lane] : -1;
    int rank = 0;
    for (int i = 0; i < seqs; ++i) {
      const int other = __builtin_amdgcn_readlane(own, i);
      rank += other > own || (other == own && i < lane);
    }
    if (lane < seqs) order[rank] = lane;
  }
  int s = -1;  // the last sequence that starts at or before this chunk
  for (int i = 0; i < seqs; i += 64) {
    const int k = i + lane;
    s += __popcll(__ballot(k < seqs && chunk_base(cu_seqlens[min(k, seqs - 1)], k) <= chunk));
  }
  if (s < 0) return;
  const int first = cu_seqlens[s], end = cu_seqlens[s + 1];
  const int t0 = first + (chunk - chunk_base(first, s)) * CQ;
  if (t0 < first || t0 >= end) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, g = lane >> 4;
  const int per = heads / groups;
  const int parts = cdiv(per, HEADS_PER_BLOCK);
  const int grp = blockIdx.y / parts;
  const int h0 = grp * per + blockIdx.y % parts * HEADS_PER_BLOCK;
  const int h_end = min(h0 + HEADS_PER_BLOCK, (grp + 1) * per);
  const int inner = heads * P;
  const long channels = inner + 2L * groups * N;

  // rows through LDS: as fragments straight from memory, 16 rows to a load with
  // neighbouring lanes in different ones, they come at a quarter of the rate
#pragma unroll
  for (int i = 0; i < CQ * NP / 4 / DT; ++i) {
    const int e = threadIdx.x + i * DT;
    const int t = e / (NP / 4), n = e % (NP / 4) * 4;
    const bool ok = t0 + t < end && n < N;
    const float* row = xbc + (t0 + t) * channels + inner + grp * N + n;
    const f32x4s zero = f32x4s{0.f, 0.f, 0.f, 0.f};
    *reinterpret_cast<f32x4s*>(Bs + t * RS + n) =
        ok ? *reinterpret_cast<const f32x4s*>(row) : zero;
    *reinterpret_cast<f32x4s*>(Cs + t * RS + n) =
        ok ? *reinterpret_cast<const f32x4s*>(row + groups * N) : zero;
  }
  __syncthreads();

  f32x4s cb[NG];  // B_s . C_t: row s, column t
#pragma unroll
  for (int i = 0; i < NG; ++i) {
    if (wave + i * NW >= CTILES) continue;
    int tb, sb;
    chunk_tile(wave + i * NW, tb, sb);
    const float* cr = Cs + (tb * 16 + col) * RS + g * 4;
    const float* br = Bs + (sb * 16 + col) * RS + g * 4;
    // eight chains: fewer roundings in a row than one sum over the states
    f32x4s acc[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) acc[r] = f32x4s{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const f32x4s c4 = *reinterpret_cast<const f32x4s*>(cr + b * 16);
      const f32x4s b4 = *reinterpret_cast<const f32x4s*>(br + b * 16);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        f32x4s& to = acc[r + (b & 1) * 4];
        to = mfma4(b4[r], c4[r], to);
      }
    }
    cb[i] = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
  }

  for (int hb = h0; hb < h_end; hb += NW) {
    __syncthreads();
    if (hb + wave < h_end) {
      const int h = hb + wave;
      // finite where exp leaves the range: differences of infinite running sums
      // would be NaN where the decay is 0
      float A = -expf(a_log[h]);
      if (A < -FLT_MAX) A = -FLT_MAX;
      const long i = (long)min(t0 + lane, end - 1) * dt_stride + h;
      const float v =
          (dt_raw_f32 ? dt_raw_f32[i] : bf16_bits_to_float(dt_raw_bf16[i])) + dt_bias[h];
      // softplus without a clamp; log1p(exp(v)) is v itself past v ~ 30.
      // Rows past the portion: dt 0, so they change nothing
      const float dt = t0 + lane < end ? (v > 30.f ? v : log1pf(expf(v))) : 0.f;
      double c = (double)A * dt * 1.4426950408889634;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const double o = __shfl_up(c, off, 64);
        if (lane >= off) c += o;
      }
      const double last = __shfl(c, 63, 64);
      cum[wave][lane] = c;
      dts[wave][lane] = dt;
      ChunkWork& to = work[(long)chunk * heads + h];
      to.grow[lane] = __builtin_amdgcn_exp2f((float)c);
      to.left[lane] = dt * __builtin_amdgcn_exp2f((float)(last - c));
    }
    __syncthreads();
    for (int k = 0; k < NW && hb + k < h_end; ++k) {
      ChunkWork& to = work[(long)chunk * heads + hb + k];
#pragma unroll
      for (int i = 0; i < NG; ++i) {
        if (wave + i * NW >= CTILES) continue;
        int tb, sb;
        chunk_tile(wave + i * NW, tb, sb);
        const int t = tb * 16 + col;
        f32x4s m;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int u = sb * 16 + g * 4 + r;
          const float d = (float)(cum[k][t] - cum[k][u]);
          // (later tokens: whatever it is, it is not taken)
          const float e = cb[i][r] * __builtin_amdgcn_exp2f(d) * dts[k][u];
          m[r] = u <= t ? e : 0.f;
        }
        to.m[wave + i * NW][lane] = m;
      }
    }
  }
}

template <int NB, int CB>  // blocks of 16 states and columns
__global__ void __launch_bounds__(ST, 2) ssd_chain_kernel(
    float* __restrict__ y, const float* __restrict__ xbc, const ChunkWork* __restrict__ work,
    const int* __restrict__ order, const float* __restrict__ d_skip, float* __restrict__ state,
    const long* __restrict__ positions, const int* __restrict__ cu_seqlens,
    const int* __restrict__ slots, int heads, int groups, int P, int N) {
  constexpr int NW = ST / 64;
  constexpr int NP = NB * 16, PB = CB * 16;
  constexpr int RS = NP + 4;  // B and state rows: 4 rows apart fall 16 banks apart
  constexpr int XS = PB + 4;
  constexpr int NH = NB / NW;           // state blocks of a wave
  constexpr int NV = CQ * NP / 4 / ST;  // float4 per thread of a B tile
  constexpr int XV = CQ * PB / 4 / ST;
  static_assert(NH * NW == NB && XV * ST * 4 == CQ * PB && CQ == 16 * NW, "tile");
  __shared__ __attribute__((aligned(16))) float Bs[CQ * RS];
  __shared__ __attribute__((aligned(16))) float Xs[CQ * XS];
  __shared__ __attribute__((aligned(16))) float Ss[PB * RS];  // by column
  __shared__ __attribute__((aligned(16))) float left[CQ];

  const int s = order ? order[blockIdx.z] : blockIdx.z, h = blockIdx.y;
  const int first = cu_seqlens[s];
  const int len = cu_seqlens[s + 1] - first;
  if (len <= 0) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int p0 = blockIdx.x * PB;
  const int grp = h / (heads / groups);
  const int inner = heads * P;
  const int channels = inner + 2 * groups * N;
  const float Dh = d_skip[h];
  const f32x4s zero = f32x4s{0.f, 0.f, 0.f, 0.f};
  float* sp = state + ((slots[s] * (long)heads + h) * P + p0) * N;

  // byte offsets within a chunk's rows: of B, of x, of C (this wave's tokens)
  const unsigned int row4 = (unsigned int)channels * 4;
  const int bn = threadIdx.x % (NP / 4) * 4, xn = threadIdx.x % (PB / 4) * 4;
  const unsigned int b_at = bn < N ? threadIdx.x / (NP / 4) * row4 + bn * 4 : OUTSIDE;
  const unsigned int x_at =
      p0 + xn < P ? threadIdx.x / (PB / 4) * row4 + xn * 4 : OUTSIDE;
  const int c_n = (threadIdx.x & 63) / 16 * 4;
  const unsigned int c_at = (wave * 16 + (threadIdx.x & 15)) * row4 + c_n * 4;
  const float* seq_rows = xbc + (long)first * channels;
  const ChunkWork* seq_work = work + (long)chunk_base(first, s) * heads + h;

  f32x4s rB[NV], rX[XV], rC[NB], rM[NW], rE;
  float rL = 0.f, keep = 0.f, keep_next;
  auto fetch_rows = [&](int t0) {
    const float* rows = seq_rows + (long)t0 * channels;
    const unsigned int last = (unsigned int)(min(len - t0, CQ) - 1) * row4;
#pragma unroll
    for (int i = 0; i < NV; ++i)
      rB[i] = load_or_zero(rows + inner + grp * N, last + N * 4,
                           b_at + i * (ST / (NP / 4)) * row4);
#pragma unroll
    for (int i = 0; i < XV; ++i)
      rX[i] = load_or_zero(rows + h * P + p0, last + (P - p0) * 4,
                           x_at + i * (ST / (PB / 4)) * row4);
    const ChunkWork& w = seq_work[(long)(t0 / CQ) * heads];
    rL = w.left[threadIdx.x % CQ];
    keep_next = w.grow[CQ - 1];
  };
  auto fetch_c = [&](int t0) {
    const float* rows = seq_rows + (long)t0 * channels + inner + (groups + grp) * N;
    const unsigned int last = (unsigned int)(min(len - t0, CQ) - 1) * row4;
#pragma unroll
    for (int b = 0; b < NB; ++b)
      rC[b] = load_or_zero(rows, last + N * 4, c_n + b * 16 < N ? c_at + b * 64 : OUTSIDE);
  };
  auto fetch_products = [&](int t0) {
    const ChunkWork& w = seq_work[(long)(t0 / CQ) * heads];
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int sb = 0; sb < NW; ++sb)
      rM[sb] = w.m[wave * (wave + 1) / 2 + min(sb, wave)][lane];
    rE = *reinterpret_cast<const f32x4s*>(w.grow + wave * 16 + lane / 16 * 4);
  };

  f32x4s S[NH][CB];
  {
    const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
    const bool fresh = positions[first] == 0;
#pragma unroll
    for (int b = 0; b < NH; ++b)
#pragma unroll
      for (int k = 0; k < CB; ++k) {
        const int n = (wave * NH + b) * 16 + g * 4, c = k * 16 + col;
        S[b][k] = (!fresh && p0 + c < P && n < N)
                      ? *reinterpret_cast<const f32x4s*>(sp + (long)c * N + n)
                      : zero;
      }
  }

  // (in the loop's order, which its waits count by)
  fetch_rows(0);
  __builtin_amdgcn_sched_barrier(0);
  fetch_c(0);
  __builtin_amdgcn_sched_barrier(0);
  fetch_products(0);
  __builtin_amdgcn_sched_barrier(0);
  for (int t0 = 0; t0 < len; t0 += CQ) {
    const int cnt = min(CQ, len - t0);
    // (the last chunk fetches itself again: were its loads left out, the waits for
    // the others would have to assume so in every chunk)
    const int next = t0 + CQ < len ? t0 + CQ : t0;
    // (lane numbers that the compiler takes for new ones: it keeps every address of
    // the chunk in a register from before the loop otherwise, more than there are)
    unsigned int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, col = lane & 15, g = lane >> 4;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const unsigned int e = tid + i * ST;
      *reinterpret_cast<f32x4s*>(Bs + e / (NP / 4) * RS + e % (NP / 4) * 4) = rB[i];
    }
#pragma unroll
    for (int i = 0; i < XV; ++i) {
      const unsigned int e = tid + i * ST;
      *reinterpret_cast<f32x4s*>(Xs + e / (PB / 4) * XS + e % (PB / 4) * 4) = rX[i];
    }
    if (wave == 0) left[lane] = rL;
    keep = keep_next;
#pragma unroll
    for (int b = 0; b < NH; ++b)
#pragma unroll
      for (int k = 0; k < CB; ++k)
        *reinterpret_cast<f32x4s*>(Ss + (k * 16 + col) * RS + (wave * NH + b) * 16 + g * 4) =
            S[b][k];
    __syncthreads();
    fetch_rows(next);
    __builtin_amdgcn_sched_barrier(0);

    // LDS reads go a step ahead of the products that want them, 8 or 16 products of
    // 32 cycles: left to itself the compiler reads each operand as it is wanted
    f32x4s X[4][CB];  // tokens 16 tb + 4 g + r, this lane's columns
    {
      const float* xrow = Xs + g * 4 * XS + col;
#pragma unroll
      for (int tb = 0; tb < 4; ++tb)
#pragma unroll
        for (int k = 0; k < CB; ++k)
#pragma unroll
          for (int r = 0; r < 4; ++r) X[tb][k][r] = xrow[(tb * 16 + r) * XS + k * 16];
    }

    // ---- what the state at the chunk's start contributes to this wave's tokens ----
    f32x4s Y[CB][4];  // four chains: fewer roundings in a row
#pragma unroll
    for (int k = 0; k < CB; ++k)
#pragma unroll
      for (int r = 0; r < 4; ++r) Y[k][r] = zero;
    f32x4s s4[2][CB];
    auto states = [&](int b) {
#pragma unroll
      for (int k = 0; k < CB; ++k)
        s4[b & 1][k] =
            *reinterpret_cast<const f32x4s*>(Ss + (k * 16 + col) * RS + b * 16 + g * 4);
    };
    states(0);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (b + 1 < NB) states(b + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int k = 0; k < CB; ++k) Y[k][r] = mfma4(rC[b][r], s4[b & 1][k][r], Y[k][r]);
      __builtin_amdgcn_sched_barrier(0);
    }
    fetch_c(next);
    __builtin_amdgcn_sched_barrier(0);

    // ---- and the chunk's own tokens ----
#pragma unroll
    for (int k = 0; k < CB; ++k) {
      f32x4s acc[4], x = zero;  // x ends as this wave's tokens' own
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] = zero;
#pragma unroll
      for (int sb = 0; sb < NW; ++sb) {
        if (sb > wave) continue;
        x = X[sb][k];
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = mfma4(rM[sb][r], x[r], acc[r]);
      }
      f32x4s z = (acc[0] + acc[1]) + (acc[2] + acc[3]);
      const f32x4s past = ((Y[k][0] + Y[k][1]) + (Y[k][2] + Y[k][3])) * rE;
      z += past;
      // The products above take later tokens of the tile with weight 0, which
      // is no 0 if their x is infinite or NaN: such sums are formed again, from
      // the tokens up to each row's own only.
      const float size = fabsf(z[0]) + fabsf(z[1]) + fabsf(z[2]) + fabsf(z[3]);
      if (__any(!(size < INFINITY))) {
        const ChunkWork& w = seq_work[(long)(t0 / CQ) * heads];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int t = g * 4 + r;
          float sum = 0.f;
          for (int u = 0; u <= wave * 16 + t; ++u)
            sum = fmaf(w.m[wave * (wave + 1) / 2 + u / 16][u % 16 / 4 * 16 + t][u % 4],
                       Xs[u * XS + k * 16 + col], sum);
          z[r] = sum + past[r];
        }
      }
      float* yrows = y + (long)(first + t0) * inner + h * P + p0;
      const unsigned int ybytes = ((cnt - 1) * inner + (P - p0)) * 4;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const unsigned int at = ((wave * 16 + g * 4 + r) * inner + k * 16 + col) * 4;
        store_or_drop(yrows, ybytes, p0 + k * 16 + col < P ? at : OUTSIDE, z[r] + Dh * x[r]);
      }
    }
    fetch_products(next);
    __builtin_amdgcn_sched_barrier(0);

    // ---- the state moves on ----
    f32x4s w4[2], b4[2][NH];  // of a block of 16 tokens: weights, B by token
    auto tokens = [&](int tb) {
      w4[tb & 1] = *reinterpret_cast<const f32x4s*>(left + tb * 16 + g * 4);
      const float* brow = Bs + (tb * 16 + g * 4) * RS + wave * NH * 16 + col;
#pragma unroll
      for (int b = 0; b < NH; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) b4[tb & 1][b][r] = brow[r * RS + b * 16];
    };
    tokens(0);
#pragma unroll
    for (int b = 0; b < NH; ++b)
#pragma unroll
      for (int k = 0; k < CB; ++k) S[b][k] *= keep;
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
      if (tb < 3) tokens(tb + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < CB; ++k) X[tb][k] *= w4[tb & 1];
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int k = 0; k < CB; ++k)
#pragma unroll
          for (int b = 0; b < NH; ++b)
            S[b][k] = mfma4(b4[tb & 1][b][r], X[tb][k][r], S[b][k]);
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();  // the chunk's tiles are consumed
  }
  const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
#pragma unroll
  for (int b = 0; b < NH; ++b)
#pragma unroll
    for (int k = 0; k < CB; ++k) {
      const int n = (wave * NH + b) * 16 + g * 4, c = k * 16 + col;
      if (p0 + c < P && n < N) *reinterpret_cast<f32x4s*>(sp + (long)c * N + n) = S[b][k];
    }
}

}  // namespace

// bytes that the scan in chunks takes for what needs no state, and an order of the
// sequences behind it
static long chunk_work_bytes(int tokens, int num_seqs, int heads) {
  return ((long)tokens / CQ + num_seqs) * heads * (long)sizeof(ChunkWork);
}
constexpr int MOST_ORDERED = 64;
extern "C" long ks_ssd_work_bytes(int tokens, int num_seqs, int heads) {
  return chunk_work_bytes(tokens, num_seqs, heads) + MOST_ORDERED * (long)sizeof(int);
}

extern "C" hipError_t ks_causal_conv_silu(
    void* out, const void* in, long in_stride, const void* w, const void* bias,
    void* conv_state, const void* positions, const void* seq_of_token,
    const void* cu_seqlens, const void* slots, int tokens, int num_seqs,
    int channels, int taps, int silu, int is_f32, int whole_portions,
    hipStream_t stream) {
  if (tokens == 0) return hipSuccess;
  if (taps < 1 || taps > MAX_TAPS) return hipErrorInvalidValue;
  dim3 grid(cdiv(channels, 256), tokens);
  dim3 grid_u(cdiv(channels, 256), num_seqs);
  const int esz = is_f32 ? 4 : 2;
  // 4-channel vectors need every row start on a 4-element boundary
  const bool vec = channels % 4 == 0 && in_stride % 4 == 0 &&
                   ((uintptr_t)in % (4 * esz)) == 0 &&
                   ((uintptr_t)conv_state % (4 * esz)) == 0 &&
                   ((uintptr_t)out % 16) == 0 && ((uintptr_t)bias % 16) == 0 &&
                   taps >= 2 && taps <= 4;
  const bool longer = (long)tokens * channels > CONV_LONG;
  dim3 grid_v(cdiv(channels / 4, 256),
              cdiv(tokens, longer ? CONV_TT_LONG : CONV_TT));
#define CONV_ARGS(TT)                                                         \
  (float*)out, (const TT*)in, in_stride, (const float*)w, (const float*)bias, \
      (const TT*)conv_state, (const long*)positions,                          \
      (const int*)seq_of_token, (const int*)cu_seqlens, (const int*)slots
  if (vec && whole_portions) {
    const dim3 grid_s(cdiv(channels / 4, 256), num_seqs);
#define CONV_SEQ_K(TT, K)                                                     \
  hipLaunchKernelGGL((causal_conv_silu_seq_kernel<TT, K>), grid_s, dim3(256), \
                     0, stream, (float*)out, (const TT*)in, in_stride,        \
                     (const float*)w, (const float*)bias, (TT*)conv_state,    \
                     (const long*)positions, (const int*)cu_seqlens,          \
                     (const int*)slots, channels, silu)
#define CONV_SEQ(TT)                                                          \
  do {                                                                        \
    if (taps == 2) CONV_SEQ_K(TT, 2);                                         \
    else if (taps == 3) CONV_SEQ_K(TT, 3);                                    \
    else CONV_SEQ_K(TT, 4);                                                   \
  } while (0)
    if (is_f32) CONV_SEQ(float);
    else CONV_SEQ(short);
    HIP_CHECK_KERNEL();
    return hipSuccess;
  }
#define CONV_VEC_N(TT, K, N)                                                  \
  hipLaunchKernelGGL((causal_conv_silu_vec4_kernel<TT, K, N>), grid_v,        \
                     dim3(256), 0, stream, CONV_ARGS(TT), tokens, channels, silu)
#define CONV_VEC_K(TT, K)                        \
  do {                                           \
    if (longer) CONV_VEC_N(TT, K, CONV_TT_LONG); \
    else CONV_VEC_N(TT, K, CONV_TT);             \
  } while (0)
#define CONV_VEC(TT)                                                          \
  do {                                                                        \
    if (taps == 2) CONV_VEC_K(TT, 2);                                         \
    else if (taps == 3) CONV_VEC_K(TT, 3);                                    \
    else CONV_VEC_K(TT, 4);                                                   \
  } while (0)
  if (is_f32) {
    if (vec) CONV_VEC(float);
    else
      hipLaunchKernelGGL(causal_conv_silu_kernel<float>, grid, dim3(256), 0,
                         stream, CONV_ARGS(float), channels, taps, silu);
    if (taps > 1)
      hipLaunchKernelGGL(conv_state_update_kernel<float>, grid_u, dim3(256), 0,
                         stream, (float*)conv_state, (const float*)in,
                         in_stride, (const long*)positions,
                         (const int*)cu_seqlens, (const int*)slots, channels,
                         taps);
  } else {
    if (vec) CONV_VEC(short);
    else
      hipLaunchKernelGGL(causal_conv_silu_kernel<short>, grid, dim3(256), 0,
                         stream, CONV_ARGS(short), channels, taps, silu);
    if (taps > 1)
      hipLaunchKernelGGL(conv_state_update_kernel<short>, grid_u, dim3(256), 0,
                         stream, (short*)conv_state, (const short*)in,
                         in_stride, (const long*)positions,
                         (const int*)cu_seqlens, (const int*)slots, channels,
                         taps);
  }
  HIP_CHECK_KERNEL();
  return hipSuccess;
}

#define SSD_LAUNCH(RR, PCC)                                                   \
  hipLaunchKernelGGL((ssd_scan_kernel<RR, PCC>), grid, dim3(256), smem,       \
                     stream, (float*)y, (const float*)xbc,                    \
                     dt_is_f32 ? (const float*)dt_raw : nullptr,              \
                     dt_is_f32 ? nullptr : (const short*)dt_raw, dt_stride,   \
                     (const float*)dt_bias, (const float*)a_log,              \
                     (const float*)d_skip, (float*)state,                     \
                     (const long*)positions, (const int*)cu_seqlens,          \
                     (const int*)slots, heads, groups, P, N)

#define SSD_LAUNCH_R(RR)                                                      \
  do {                                                                        \
    if (pc == 1) SSD_LAUNCH(RR, 1);                                           \
    else if (pc == 2) SSD_LAUNCH(RR, 2);                                      \
    else SSD_LAUNCH(RR, 4);                                                   \
  } while (0)

extern "C" hipError_t ks_ssd_scan(void* y, const void* xbc, const void* dt_raw,
                                  long dt_stride, int dt_is_f32,
                                  const void* dt_bias, const void* a_log,
                                  const void* d_skip, void* state,
                                  const void* positions,
                                  const void* cu_seqlens, const void* slots,
                                  int tokens, int num_seqs, int heads,
                                  int groups, int P, int N, int chunks,
                                  void* work, hipStream_t stream) {
  if (num_seqs == 0) return hipSuccess;
  if (groups <= 0 || heads % groups != 0 || N < 1 || N > 256)
    return hipErrorInvalidValue;
  if (chunks && N % 4 == 0 && N <= 128 && P % 4 == 0 &&
      (((uintptr_t)xbc | (uintptr_t)state) & 15) == 0) {
#define SSD_DT                                                                \
  dt_is_f32 ? (const float*)dt_raw : nullptr,                                 \
      dt_is_f32 ? nullptr : (const short*)dt_raw, dt_stride,                  \
      (const float*)dt_bias, (const float*)a_log
    if (!work) {
      const dim3 cgrid(cdiv(P, 64), heads, num_seqs);
#define SSD_CHUNK(nb)                                                         \
  hipLaunchKernelGGL((ssd_chunk_kernel<nb>), cgrid, dim3(CT), 0, stream,      \
                     (float*)y, (const float*)xbc, SSD_DT,                    \
                     (const float*)d_skip, (float*)state,                     \
                     (const long*)positions, (const int*)cu_seqlens,          \
                     (const int*)slots, heads, groups, P, N)
      if (N <= 32) SSD_CHUNK(2);
      else if (N <= 64) SSD_CHUNK(4);
      else SSD_CHUNK(8);
#undef SSD_CHUNK
      HIP_CHECK_KERNEL();
      return hipSuccess;
    }
    if (((uintptr_t)work & 15) != 0) return hipErrorInvalidValue;
    const dim3 pgrid((unsigned)(tokens / CQ + num_seqs),
                     groups * cdiv(heads / groups, HEADS_PER_BLOCK));
    // 32 columns a block, or 16 where the chip has room for twice the blocks
    // (64 heads of 64 columns, 8000 tokens of 1 / 2 / 4 sequences: 568 / 398, 157 /
    // 158, 260 / 327 us)
    const int cb =
        chunks > 2 ? chunks - 2 : P <= 16 || cdiv(P, 32) * (long)heads * num_seqs <= 192 ? 1 : 2;
    const dim3 cgrid(cdiv(P, 16 * cb), heads, num_seqs);
    // The longest portions first where the blocks come to two rounds at most: the long
    // ones then share their units with the short ones (6 portions of 200 to 3000 tokens
    // 324 -> 282 us); more rounds even out by themselves.
    int* const order =
        num_seqs > 1 && num_seqs <= MOST_ORDERED &&
                cgrid.x * (long)cgrid.y * cgrid.z <= 4L * 256
            ? (int*)((char*)work + chunk_work_bytes(tokens, num_seqs, heads))
            : nullptr;
#define SSD_CHAIN(nb, cbs)                                                    \
  hipLaunchKernelGGL((ssd_chain_kernel<nb, cbs>), cgrid, dim3(ST), 0, stream, \
                     (float*)y, (const float*)xbc, (const ChunkWork*)work,    \
                     (const int*)order, (const float*)d_skip, (float*)state,                     \
                     (const long*)positions, (const int*)cu_seqlens,          \
                     (const int*)slots, heads, groups, P, N)
#define SSD_CHAINS(nb)                                                        \
  do {                                                                        \
    hipLaunchKernelGGL((ssd_decays_kernel<nb>), pgrid, dim3(DT), 0, stream,   \
                       (ChunkWork*)work, order, (const float*)xbc, SSD_DT,    \
                       (const int*)cu_seqlens, num_seqs, heads, groups, P,    \
                       N);                                                    \
    HIP_CHECK_KERNEL();                                                       \
    if (cb == 1) SSD_CHAIN(nb, 1);                                            \
    else SSD_CHAIN(nb, 2);                                                    \
  } while (0)
    if (N <= 64) SSD_CHAINS(4);
    else SSD_CHAINS(8);
#undef SSD_CHAINS
#undef SSD_CHAIN
#undef SSD_DT
    HIP_CHECK_KERNEL();
    return hipSuccess;
  }
  // A token or two per sequence: whole state rows by 16-byte lanes (us, token by
  // token in chunks of 16 -> this, 64 heads of 64 x 128, states not in a cache:
  // 128 x 1 token 162 -> 105, 128 x 2 164 -> 108, 4 of 1 to 5 18 -> 13). One long
  // portion among them is walked at 1.0 to 1.7 us per token here and there, and
  // the rule keeps it to about as many tokens as there are sequences, whose
  // states cost more than the walk gains there: 127 x 1 + 100 254 -> 214, 127 x 1
  // + 129 277 -> 250, 399 x 1 + 401 817 -> 764, 1019 x 1 + 1020 2060 -> 1920
  // (with 500 beside 127 it would be 612 -> 655, past the rule)
  if (tokens <= 2L * num_seqs && (N == 64 || N == 128) && P % 64 == 0 &&
      (((uintptr_t)xbc | (uintptr_t)state) & 15) == 0) {
    const dim3 sgrid(P / 64, heads, num_seqs);
#define SSD_STEP(nl)                                                          \
  hipLaunchKernelGGL((ssd_step_kernel<nl>), sgrid, dim3(256), 0, stream,      \
                     (float*)y, (const float*)xbc,                            \
                     dt_is_f32 ? (const float*)dt_raw : nullptr,              \
                     dt_is_f32 ? nullptr : (const short*)dt_raw, dt_stride,   \
                     (const float*)dt_bias, (const float*)a_log,              \
                     (const float*)d_skip, (float*)state,                     \
                     (const long*)positions, (const int*)cu_seqlens,          \
                     (const int*)slots, heads, groups, P)
    if (N == 64) SSD_STEP(16);
    else SSD_STEP(32);
#undef SSD_STEP
    HIP_CHECK_KERNEL();
    return hipSuccess;
  }
  // columns per lane: a block covers up to 64 columns of one head; wide
  // state rows (R = 16) keep two columns so the state stays in registers
  const int R = cdiv(N, 16);
  int pc = P > 32 ? 4 : (P > 16 ? 2 : 1);
  if (R > 8 && pc > 2) pc = 2;
  const int xs = 16 * pc;
  const size_t smem = sizeof(float) * ((size_t)SCAN_TC * (2 * N + 2 * xs + 2));
  dim3 grid(cdiv(P, xs), heads, num_seqs);
  if (R <= 1) SSD_LAUNCH_R(1);
  else if (R <= 2) SSD_LAUNCH_R(2);
  else if (R <= 3) SSD_LAUNCH_R(3);
  else if (R <= 4) SSD_LAUNCH_R(4);
  else if (R <= 6) SSD_LAUNCH_R(6);
  else if (R <= 8) SSD_LAUNCH_R(8);
  else SSD_LAUNCH_R(16);
  HIP_CHECK_KERNEL();
  return hipSuccess;
}
