// Depthwise causal short convolution over [shared prefix taps || beam suffix].
//
// Replaces src/kadllm/ops.py:166-226 and src/kadllm/kernels/causal_conv1d.py:10-78.
// HBM-bound: each output element reads its input once; the request-sized
// prefix taps (state[b, c, history-3 ..]) and the weights are read by every
// beam of the request and stay in L2.  Rounding follows the reference torch
// path: the convolution result is rounded to the tensor dtype, then SiLU is
// applied and rounded again (for fp32 both roundings are exact).  The bf16
// kernels (decode and prefill) take SiLU with the hardware reciprocal
// (silu_fast: they are VALU-bound and the result is rounded to bf16); fp16 and
// fp32 tensors keep the IEEE exp and divide.
//
// Three paths: a vectorised one when channels are contiguous in x and out (the
// [rows, T, C] layout produced by the projection GEMM), a vectorised one for the
// reference's contiguous [BW, C, T] layout, both in 16-byte words of any of the
// three types, and a scalar one for any other strides and widths.

#include <algorithm>

#include "kad_common.h"

namespace {

template <typename T>
__device__ __forceinline__ float ld(const T* p) { return Elem<T>::to_f(*p); }

// SiLU in the dtype's precision: the hardware reciprocal for bf16 outputs, the
// IEEE exp and divide (torch's silu) for fp16 and fp32
template <typename T>
__device__ __forceinline__ float silu_for(float x) {
  if constexpr (Elem<T>::code == KAD_DTYPE_BF16) return silu_fast(x);
  else return x / (1.0f + expf(-x));
}

template <typename T>
__global__ __launch_bounds__(256) void conv_suffix_scalar(
    const T* __restrict__ x, int64_t sx_n, int64_t sx_c, int64_t sx_t,
    const T* __restrict__ state, int64_t ss_b, int64_t ss_c, int64_t ss_t, int history,
    const T* __restrict__ w, int width, const T* __restrict__ bias, T* __restrict__ out,
    int64_t so_n, int64_t so_c, int64_t so_t, int W, int C, int T_, int64_t total, int silu) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const int c = (int)(idx % C);
  const int64_t n = idx / C;
  const int64_t b = n / W;
  if (width > 4) {
    // wide kernels: each output reads its window straight from the prefix
    // taps and the suffix, taps in weight order as the width-4 path
    const float bv = bias ? ld(bias + c) : 0.f;
    for (int t = 0; t < T_; ++t) {
      float acc = bv;
      for (int i = 0; i < width; ++i) {
        const int p = t + i - (width - 1);  // < 0: prefix tap history + p
        const float xv = p < 0 ? ld(state + b * ss_b + (int64_t)c * ss_c + (int64_t)(history + p) * ss_t)
                               : ld(x + n * sx_n + (int64_t)c * sx_c + (int64_t)p * sx_t);
        acc += ld(w + (int64_t)c * width + i) * xv;
      }
      float y = round_to_dtype(acc, Elem<T>::code);
      if (silu) y = silu_for<T>(y);
      out[n * so_n + (int64_t)c * so_c + (int64_t)t * so_t] = Elem<T>::from_f(y);
    }
    return;
  }
  float win[4] = {0.f, 0.f, 0.f, 0.f};  // win[3] is the newest tap
  float wt[4] = {0.f, 0.f, 0.f, 0.f};
  for (int i = 0; i < width; ++i) wt[4 - width + i] = ld(w + (int64_t)c * width + i);
  for (int i = 0; i < width - 1; ++i)
    win[4 - (width - 1) + i] = ld(state + b * ss_b + (int64_t)c * ss_c +
                                  (int64_t)(history - (width - 1) + i) * ss_t);
  const float bv = bias ? ld(bias + c) : 0.f;
  for (int t = 0; t < T_; ++t) {
    win[0] = win[1];
    win[1] = win[2];
    win[2] = win[3];
    win[3] = ld(x + n * sx_n + (int64_t)c * sx_c + (int64_t)t * sx_t);
    float acc = bv;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc += wt[i] * win[i];
    float y = round_to_dtype(acc, Elem<T>::code);
    if (silu) y = silu_for<T>(y);
    out[n * so_n + (int64_t)c * so_c + (int64_t)t * so_t] = Elem<T>::from_f(y);
  }
}

// A 16-byte word of channels and the layout-independent parts of the vector
// kernels: VE channels per thread, whose weights ([C, 4]) are 64 bytes and
// whose prefix taps are 64 bytes in the model's state layout ([B, C, 4]).
template <typename T>
struct ConvVec {
  static constexpr int VE = 16 / sizeof(T);
  __device__ static __forceinline__ void unpack(const u32x4& r, float (&f)[VE]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (Elem<T>::code == KAD_DTYPE_BF16) {
        f[2 * e] = __uint_as_float(r[e] << 16);
        f[2 * e + 1] = __uint_as_float(r[e] & 0xffff0000u);
      } else if constexpr (Elem<T>::code == KAD_DTYPE_F16) {
        f[2 * e] = (float)__builtin_bit_cast(_Float16, (uint16_t)(r[e] & 0xffffu));
        f[2 * e + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(r[e] >> 16));
      } else {
        f[e] = __uint_as_float(r[e]);
      }
    }
  }
  // conv results to outputs: rounded, SiLU, rounded (bf16 pairs as one packed
  // conversion each, the same bits)
  __device__ static __forceinline__ u32x4 finish(const float (&acc)[VE], bool silu) {
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (Elem<T>::code == KAD_DTYPE_BF16) {
        uint32_t p = pack_bf16x2(acc[2 * e], acc[2 * e + 1]);
        if (silu)
          p = pack_bf16x2(silu_fast(__uint_as_float(p << 16)),
                          silu_fast(__uint_as_float(p & 0xffff0000u)));
        o[e] = p;
      } else if constexpr (Elem<T>::code == KAD_DTYPE_F16) {
        uint32_t p = 0;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          float y = (float)(_Float16)acc[2 * e + h];
          if (silu) y = silu_for<T>(y);
          p |= (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)y) << (16 * h);
        }
        o[e] = p;
      } else {
        o[e] = __float_as_uint(silu ? silu_for<T>(acc[e]) : acc[e]);
      }
    }
    return o;
  }
  // VE channels x 4 from 64 contiguous bytes
  __device__ static __forceinline__ void load4(const T* p, float (&f)[VE][4]) {
    float g[VE];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      unpack(((const u32x4*)p)[j], g);
#pragma unroll
      for (int e = 0; e < VE; ++e) f[(j * VE + e) / 4][(j * VE + e) % 4] = g[e];
    }
  }
  // the last 3 taps of channels c0 .. c0 + VE - 1
  __device__ static __forceinline__ void taps(const T* sb, int c0, int64_t ss_c, int64_t ss_t,
                                              int history, float (&tap)[VE][3]) {
    if (ss_t == 1 && ss_c == 4 && history == 4 && ((uintptr_t)sb % 16) == 0) {
      float f[VE][4];
      load4(sb + (int64_t)c0 * 4, f);
#pragma unroll
      for (int ch = 0; ch < VE; ++ch)
#pragma unroll
        for (int i = 0; i < 3; ++i) tap[ch][i] = f[ch][i + 1];
    } else {
#pragma unroll
      for (int ch = 0; ch < VE; ++ch)
#pragma unroll
        for (int i = 0; i < 3; ++i)
          tap[ch][i] = Elem<T>::to_f(sb[(c0 + ch) * ss_c + (history - 3 + i) * ss_t]);
    }
  }
};

// Channels contiguous (a projection's rows): VE channels per thread, up to
// kConvBeams beams of one request per thread (the request's weights and prefix
// taps are loaded once); width 4 (3 taps), any T.  Grid: x = request x beam
// group, y = channel groups of 256 threads, z = runs of kConvRun tokens of
// suffixes longer than 4 (an fp32 model's whole prompts, which one thread per
// channel would walk; longer runs where a grid does not hold as many).  The next (beam, token) row is loaded before the current
// one is computed so that every thread keeps one 16-byte load in flight.
constexpr int kConvBeams = 8, kConvRun = 16;

// TT > 0: the suffix length fixed at compile time (the search's one- to
// four-token suffixes), so the (beam, token) of each step needs no division
template <typename T, int TT>
__global__ __launch_bounds__(256) void conv_suffix_vec(
    const T* __restrict__ x, int64_t sx_n, int64_t sx_t, const T* __restrict__ state,
    int64_t ss_b, int64_t ss_c, int64_t ss_t, int history, const T* __restrict__ w,
    T* __restrict__ out, int64_t so_n, int64_t so_t, int W, int C, int T_rt, int nbg, int beams,
    int run, int silu) {
  constexpr int VE = ConvVec<T>::VE;
  const int t0 = TT > 0 ? 0 : blockIdx.z * run;
  const int T_ = TT > 0 ? TT : min(run, T_rt - t0);
  const int cv = blockIdx.y * 256 + threadIdx.x;
  if (cv >= C / VE) return;
  const int c0 = cv * VE;
  const int b = blockIdx.x / nbg;
  const int j0 = (blockIdx.x % nbg) * beams;
  const int nj = min(W - j0, beams);
  const int64_t n0 = (int64_t)b * W + j0;
  const int steps = nj * T_;
  auto row = [&](int k) {
    const int j = k / T_, t = k - (k / T_) * T_;
    return x + (n0 + j) * sx_n + (int64_t)(t0 + t) * sx_t + c0;
  };
  u32x4 next = *(const u32x4*)row(0);
  float wt[VE][4], tap[VE][3];
  ConvVec<T>::load4(w + (int64_t)c0 * 4, wt);
  if (TT > 0 || t0 == 0) ConvVec<T>::taps(state + b * ss_b, c0, ss_c, ss_t, history, tap);

  float win[VE][4];
  for (int k = 0, t = 0; k < steps; ++k) {
    const u32x4 r = next;
    if (k + 1 < steps) next = *(const u32x4*)row(k + 1);
    if (t == 0) {
      if (TT > 0 || t0 == 0) {
#pragma unroll
        for (int ch = 0; ch < VE; ++ch)
#pragma unroll
          for (int i = 0; i < 3; ++i) win[ch][i + 1] = tap[ch][i];
      } else {  // the three tokens before the run
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          float f[VE];
          ConvVec<T>::unpack(*(const u32x4*)(row(k) + (int64_t)(i - 3) * sx_t), f);
#pragma unroll
          for (int ch = 0; ch < VE; ++ch) win[ch][i + 1] = f[ch];
        }
      }
    }
    float xv[VE], acc[VE];
    ConvVec<T>::unpack(r, xv);
#pragma unroll
    for (int ch = 0; ch < VE; ++ch) {
      win[ch][0] = win[ch][1];
      win[ch][1] = win[ch][2];
      win[ch][2] = win[ch][3];
      win[ch][3] = xv[ch];
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) s += wt[ch][i] * win[ch][i];
      acc[ch] = s;
    }
    const int j = k / T_;
    *(u32x4*)(out + (n0 + j) * so_n + (int64_t)(t0 + t) * so_t + c0) =
        ConvVec<T>::finish(acc, silu);
    if (++t == T_) t = 0;
  }
}

// The reference's contiguous [BW, C, T] layout (each beam's block of C * T
// elements is one contiguous run, tokens fastest): VE channels x TT tokens per
// thread are TT consecutive 16-byte words.  A wave moves its 64 TT words as
// they lie in memory and hands each lane its own TT through LDS (a lane loading
// its own words touches every line TT times: 32 x 256 beams x 6,144 channels of
// three bf16 tokens 159 us, 126 this way, 4.8 TB/s as the token-major kernel).  Lane l's words are l TT + k; bits 4 and up of a
// word's index are folded into its low ones so that the 16 lanes of an access
// hit 16 bank groups (TT = 2, 4; at 3 they do as they are).  Same grid and
// arithmetic as conv_suffix_vec; the next beam's words load meanwhile.
template <typename T, int TT>
__global__ __launch_bounds__(256) void conv_suffix_ct(
    const T* __restrict__ x, int64_t sx_n, const T* __restrict__ state, int64_t ss_b,
    int64_t ss_c, int64_t ss_t, int history, const T* __restrict__ w, T* __restrict__ out,
    int64_t so_n, int W, int C, int nbg, int beams, int silu) {
  constexpr int VE = ConvVec<T>::VE;
  __shared__ __attribute__((aligned(16))) u32x4 words[4][64 * TT];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int cw = blockIdx.y * 256 + wave * 64;  // the wave's first channel group
  const int lanes = min(64, C / VE - cw);       // its channel groups
  if (lanes <= 0) return;
  u32x4* own = words[wave];
  auto slot = [](int i) { return TT == 2 ? i ^ ((i >> 4) & 1) : (TT == 4 ? i ^ ((i >> 4) & 3) : i); };
  const int c0 = (cw + min(lane, lanes - 1)) * VE;
  const int b = blockIdx.x / nbg;
  const int j0 = (blockIdx.x % nbg) * beams;
  const int nj = min(W - j0, beams);
  const int64_t n0 = (int64_t)b * W + j0;
  const int64_t off = (int64_t)cw * VE * TT;    // the wave's words in a beam's block
  const int nw = lanes * TT;
  u32x4 next[TT];
  auto fetch = [&](int j) {
#pragma unroll
    for (int k = 0; k < TT; ++k)
      next[k] = ((const u32x4*)(x + (n0 + j) * sx_n + off))[min(k * 64 + lane, nw - 1)];
  };
  // The hardware keeps a wave's LDS accesses in order, so lanes exchange words
  // without a barrier; the compiler, to which each lane's addresses look
  // disjoint, must be told to.
  auto wave_order = [] { asm volatile("" ::: "memory"); };
  fetch(0);
  float wt[VE][4], tap[VE][3];
  ConvVec<T>::load4(w + (int64_t)c0 * 4, wt);
  ConvVec<T>::taps(state + b * ss_b, c0, ss_c, ss_t, history, tap);

  for (int j = 0; j < nj; ++j) {
    u32x4 cur[TT];
    if constexpr (TT > 1) {
#pragma unroll
      for (int k = 0; k < TT; ++k) own[slot(k * 64 + lane)] = next[k];
      wave_order();
      if (j + 1 < nj) fetch(j + 1);
#pragma unroll
      for (int k = 0; k < TT; ++k) cur[k] = own[slot(lane * TT + k)];
      wave_order();
    } else {
      cur[0] = next[0];
      if (j + 1 < nj) fetch(j + 1);
    }
    float f[TT][VE], y[TT][VE];
#pragma unroll
    for (int k = 0; k < TT; ++k) ConvVec<T>::unpack(cur[k], f[k]);
#pragma unroll
    for (int ch = 0; ch < VE; ++ch) {
      float w0 = tap[ch][0], w1 = tap[ch][1], w2 = tap[ch][2];
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        const int e = ch * TT + t;  // element index within the lane's words
        const float xv = f[e / VE][e % VE];
        float acc = 0.f;
        acc += wt[ch][0] * w0;
        acc += wt[ch][1] * w1;
        acc += wt[ch][2] * w2;
        acc += wt[ch][3] * xv;
        w0 = w1;
        w1 = w2;
        w2 = xv;
        y[e / VE][e % VE] = acc;
      }
    }
    u32x4* o = (u32x4*)(out + (n0 + j) * so_n + off);
#pragma unroll
    for (int k = 0; k < TT; ++k) cur[k] = ConvVec<T>::finish(y[k], silu);
    if constexpr (TT > 1) {
#pragma unroll
      for (int k = 0; k < TT; ++k) own[slot(lane * TT + k)] = cur[k];
      wave_order();
#pragma unroll
      for (int k = 0; k < TT; ++k) cur[k] = own[slot(k * 64 + lane)];
      wave_order();
    }
#pragma unroll
    for (int k = 0; k < TT; ++k)
      if (k * 64 + lane < nw) o[k * 64 + lane] = cur[k];
  }
}

// Prefill: causal width-4 conv + SiLU over whole prompts with zero history
// (transformers causal_conv1d_fn, modeling_qwen3_5.py:220-239), and the conv
// state the decode path reads: the last 4 pre-conv inputs of each sequence
// (cache_utils.py:1032-1070), zero-padded on the left for prompts shorter
// than 4.  Rows are tokens (row = b * L + t) with channels contiguous; each
// thread owns 8 channels of a run of kRun tokens and reads a 3-token halo.
constexpr int kRun = 16;

__global__ __launch_bounds__(256) void conv_prefill_bf16(
    const bf16_t* __restrict__ x, int64_t ldx, const bf16_t* __restrict__ w,
    bf16_t* __restrict__ out, int64_t ldo, bf16_t* __restrict__ state, int B, int L, int C,
    int silu) {
  const int C8 = C / 8;
  const int runs = (L + kRun - 1) / kRun;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)B * runs * C8) return;
  const int c0 = (int)(idx % C8) * 8;
  const int64_t br = idx / C8;
  const int run = (int)(br % runs);
  const int b = (int)(br / runs);
  const int t0 = run * kRun;
  float wt[8][4];
  {
    const u32x4* wp = (const u32x4*)(w + (int64_t)c0 * 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      u32x4 r = wp[j];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int flat = j * 8 + e * 2;
        wt[flat / 4][flat % 4] = __uint_as_float(r[e] << 16);
        wt[(flat + 1) / 4][(flat + 1) % 4] = __uint_as_float(r[e] & 0xffff0000u);
      }
    }
  }
  float win[8][4];
#pragma unroll
  for (int ch = 0; ch < 8; ++ch) win[ch][0] = win[ch][1] = win[ch][2] = win[ch][3] = 0.f;
  // halo: tokens t0-3 .. t0-1 (zero before the sequence start)
  for (int h = 3; h >= 1; --h) {
    const int t = t0 - h;
    float xv[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (t >= 0) {
      const u32x4 r = *(const u32x4*)(x + ((int64_t)b * L + t) * ldx + c0);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        xv[2 * e] = __uint_as_float(r[e] << 16);
        xv[2 * e + 1] = __uint_as_float(r[e] & 0xffff0000u);
      }
    }
#pragma unroll
    for (int ch = 0; ch < 8; ++ch) {
      win[ch][0] = win[ch][1];
      win[ch][1] = win[ch][2];
      win[ch][2] = win[ch][3];
      win[ch][3] = xv[ch];
    }
  }
  const int t_end = min(L, t0 + kRun);
  // the run's rows are all loaded before any is used (kRun loads in flight)
  u32x4 rows_in[kRun];
#pragma unroll
  for (int i = 0; i < kRun; ++i)
    rows_in[i] = *(const u32x4*)(x + ((int64_t)b * L + min(t0 + i, L - 1)) * ldx + c0);
#pragma unroll
  for (int i = 0; i < kRun; ++i) {
    const int t = t0 + i;
    if (t >= t_end) break;
    const u32x4 r = rows_in[i];
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float xv[2] = {__uint_as_float(r[e] << 16), __uint_as_float(r[e] & 0xffff0000u)};
      float acc[2];
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const int ch = e * 2 + hh;
        win[ch][0] = win[ch][1];
        win[ch][1] = win[ch][2];
        win[ch][2] = win[ch][3];
        win[ch][3] = xv[hh];
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) s += wt[ch][i] * win[ch][i];
        acc[hh] = s;
      }
      // the pair's bf16 roundings (the conv output, then the SiLU output) as
      // one packed conversion each; SiLU with the hardware reciprocal, as in
      // the decode conv kernels (within one bf16 ulp of torch's silu)
      uint32_t packed = pack_bf16x2(acc[0], acc[1]);
      if (silu)
        packed = pack_bf16x2(silu_fast(__uint_as_float(packed << 16)),
                             silu_fast(__uint_as_float(packed & 0xffff0000u)));
      o[e] = packed;
    }
    *(u32x4*)(out + ((int64_t)b * L + t) * ldo + c0) = o;
  }
  // conv state [B, C, 4]: inputs at positions L-4 .. L-1 (the run holding L-1 writes it)
  if (state && t_end == L) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int t = L - 4 + j;
#pragma unroll
      for (int ch = 0; ch < 8; ++ch) {
        const float v = t >= 0 ? bf2f(x[((int64_t)b * L + t) * ldx + c0 + ch]) : 0.f;
        state[((int64_t)b * C + c0 + ch) * 4 + j] = f2bf(v);
      }
    }
  }
}

template <typename T>
int launch_scalar(const void* x, int64_t sx_n, int64_t sx_c, int64_t sx_t, const void* state,
                  int64_t ss_b, int64_t ss_c, int64_t ss_t, int history, const void* w,
                  int width, const void* bias, void* out, int64_t so_n, int64_t so_c,
                  int64_t so_t, int B, int W, int C, int T_, int silu, hipStream_t s) {
  const int64_t total = (int64_t)B * W * C;
  hipLaunchKernelGGL((conv_suffix_scalar<T>), dim3((unsigned)kad_cdiv(total, 256)), dim3(256), 0,
                     s, (const T*)x, sx_n, sx_c, sx_t, (const T*)state, ss_b, ss_c, ss_t,
                     history, (const T*)w, width, (const T*)bias, (T*)out, so_n, so_c, so_t, W,
                     C, T_, total, silu);
  return kad_launch_status("conv_suffix_scalar");
}

// 16-byte words of channels: the vector kernels where the layout has them, the
// scalar one for other strides, widths and a bias
template <typename T>
int launch_typed(const void* x, int64_t sx_n, int64_t sx_c, int64_t sx_t, const void* state,
                 int64_t ss_b, int64_t ss_c, int64_t ss_t, int history, const void* w, int width,
                 const void* bias, void* out, int64_t so_n, int64_t so_c, int64_t so_t, int B,
                 int W, int C, int T_, int silu, hipStream_t s) {
  constexpr int VE = ConvVec<T>::VE;
  const bool words = width == 4 && bias == nullptr && C % VE == 0 && sx_n % VE == 0 &&
                     so_n % VE == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)out % 16) == 0 &&
                     ((uintptr_t)w % 16) == 0;
  // fp16's IEEE SiLU eight times a thread is its time, so below 8 M elements of
  // token-major rows more threads of one channel each take less (8 x 50 beams of
  // 6,144 channels, 1 / 2 tokens 17.4 / 19.0 us in words, 14.9 / 16.6; 4 22.2 both)
  const bool scalar16 = Elem<T>::code == KAD_DTYPE_F16 && T_ <= 4 &&
                        (int64_t)B * W * C * T_ < (8 << 20);
  // token-major rows (of one token both layouts are that)
  const bool vec = words && sx_c == 1 && so_c == 1 &&
                   (T_ == 1 || (sx_t % VE == 0 && so_t % VE == 0)) && !scalar16;
  // [BW, C, T] with each beam's C * T block contiguous (the reference's layout)
  const bool ct = words && T_ <= 4 && sx_t == 1 && sx_c == T_ && so_t == 1 && so_c == T_;
  const int groups = (int)kad_cdiv(C / VE, 256);
  // fewer beams per thread where that leaves fewer than four workgroups per CU
  int beams = kConvBeams;
  while (beams > 1 && (int64_t)B * kad_cdiv(W, beams) * groups < 1024) beams /= 2;
  const int nbg = (int)kad_cdiv(W, beams);
  if (vec) {
    KAD_REQUIRE((int64_t)B * nbg < 2147483647, "too many beams for the grid");
    const int run = (int)std::max<int64_t>(kConvRun, kad_cdiv(T_, 65535));
    const int64_t runs = T_ > 4 ? kad_cdiv(T_, run) : 1;
    const dim3 grid((unsigned)(B * nbg), (unsigned)groups, (unsigned)runs);
#define KAD_CONV_VEC(TTV)                                                                       \
  hipLaunchKernelGGL((conv_suffix_vec<T, TTV>), grid, dim3(256), 0, s, (const T*)x, sx_n, sx_t, \
                     (const T*)state, ss_b, ss_c, ss_t, history, (const T*)w, (T*)out, so_n,    \
                     so_t, W, C, T_, nbg, beams, run, silu)
    switch (T_) {
      case 1: KAD_CONV_VEC(1); break;
      case 2: KAD_CONV_VEC(2); break;
      case 3: KAD_CONV_VEC(3); break;
      case 4: KAD_CONV_VEC(4); break;
      default: KAD_CONV_VEC(0); break;
    }
#undef KAD_CONV_VEC
    return kad_launch_status("conv_suffix_vec");
  }
  if (ct) {
    KAD_REQUIRE((int64_t)B * nbg < 2147483647, "too many beams for the grid");
    const dim3 grid((unsigned)(B * nbg), (unsigned)groups);
#define KAD_CONV_CT(TTV)                                                                        \
  hipLaunchKernelGGL((conv_suffix_ct<T, TTV>), grid, dim3(256), 0, s, (const T*)x, sx_n,        \
                     (const T*)state, ss_b, ss_c, ss_t, history, (const T*)w, (T*)out, so_n, W, \
                     C, nbg, beams, silu)
    switch (T_) {
      case 1: KAD_CONV_CT(1); break;
      case 2: KAD_CONV_CT(2); break;
      case 3: KAD_CONV_CT(3); break;
      default: KAD_CONV_CT(4); break;
    }
#undef KAD_CONV_CT
    return kad_launch_status("conv_suffix_ct");
  }
  return launch_scalar<T>(x, sx_n, sx_c, sx_t, state, ss_b, ss_c, ss_t, history, w, width, bias,
                          out, so_n, so_c, so_t, B, W, C, T_, silu, s);
}

}  // namespace

extern "C" int kad_causal_conv_suffix(const void* x, int64_t sx_n, int64_t sx_c, int64_t sx_t,
                                      const void* state, int64_t ss_b, int64_t ss_c,
                                      int64_t ss_t, int history, const void* weight, int width,
                                      const void* bias, void* out, int64_t so_n, int64_t so_c,
                                      int64_t so_t, int B, int W, int C, int T, int dtype,
                                      int activation_silu, kad_stream_t stream) {
  KAD_REQUIRE(x && state && weight && out, "null pointer argument");
  KAD_REQUIRE(B > 0 && W > 0 && C > 0 && T > 0 && width > 0, "dimensions must be positive");
  if (width > 64) KAD_UNSUPPORTED("causal conv supports width <= 64, got %d", width);
  KAD_REQUIRE(history >= width - 1, "state history %d shorter than width-1", history);
  KAD_REQUIRE((int64_t)B * W * C < ((int64_t)1 << 40), "problem too large");
  hipStream_t s = (hipStream_t)stream;
#define KAD_CONV(T)                                                                            \
  return launch_typed<T>(x, sx_n, sx_c, sx_t, state, ss_b, ss_c, ss_t, history, weight, width, \
                         bias, out, so_n, so_c, so_t, B, W, C, T_, activation_silu, s)
  const int T_ = T;
  if (dtype == KAD_DTYPE_BF16) KAD_CONV(bf16_t);
  if (dtype == KAD_DTYPE_F32) KAD_CONV(float);
  if (dtype == KAD_DTYPE_F16) KAD_CONV(_Float16);
#undef KAD_CONV
  KAD_UNSUPPORTED("causal conv supports bf16, fp16 and fp32, got dtype %d", dtype);
}

extern "C" int kad_causal_conv_prefill(const void* x, int64_t ldx, const void* weight, void* out,
                                       int64_t ldo, void* state, int B, int L, int C,
                                       int activation_silu, kad_stream_t stream) {
  KAD_REQUIRE(x && weight && out, "null pointer argument");
  KAD_REQUIRE(B > 0 && L > 0 && C > 0 && C % 8 == 0, "bad dimensions (C %% 8 == 0 required)");
  KAD_REQUIRE(ldx % 8 == 0 && ldo % 8 == 0 && ((uintptr_t)x % 16) == 0 &&
                  ((uintptr_t)out % 16) == 0 && ((uintptr_t)weight % 16) == 0,
              "16-byte aligned rows required");
  const int runs = (L + kRun - 1) / kRun;
  const int64_t total = (int64_t)B * runs * (C / 8);
  hipLaunchKernelGGL(conv_prefill_bf16, dim3((unsigned)kad_cdiv(total, 256)), dim3(256), 0,
                     (hipStream_t)stream, (const bf16_t*)x, ldx, (const bf16_t*)weight,
                     (bf16_t*)out, ldo, (bf16_t*)state, B, L, C, activation_silu);
  return kad_launch_status("conv_prefill_bf16");
}
