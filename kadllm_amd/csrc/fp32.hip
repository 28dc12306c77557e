// fp32 model kernels (gfx950): the projections and row-wise layer ops of a
// Qwen3.5 model held in fp32.
//
// The reference adapter runs any float model (src/kadllm/adapters/qwen3_5.py
// wraps whatever dtype the transformers model has), and its fp32 runs are
// where it states its fixed-history accuracy (README.md:152).  The bf16 path
// of this library rounds where the transformers bf16 modules round; these
// kernels are the same layer math with no rounding at all, fp32 throughout:
//   kad_gemm_f32           C = A W^T on v_mfma_f32_16x16x4_f32 (exact fp32
//                          products, fp32 accumulation), store / residual /
//                          SwiGLU epilogues as kad_gemm_bf16
//   kad_rmsnorm_f32        x rsqrt(mean x^2 + eps) (w_offset + w)
//   kad_rmsnorm_gated_f32  w (x rsqrt(mean x^2 + eps)) silu(z) per head
//   kad_gdn_gates_f32      g = -exp(A_log) softplus(a + dt_bias), beta = sigmoid(b)
//   kad_qk_norm_rope_f32   per-head RMSNorm(1 + w), then rotate-half RoPE on
//                          the first `rot` dims with fp32 cos/sin
//   kad_embedding_f32      row gather
// They serve small fp32 models (the reference's CPU-plumbing configuration);
// the bf16 kernels serve the headline model.

#include <type_traits>

#include "kad_common.h"

namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4_t mfma16x16x4f32(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// torch's fp32 silu and sigmoid: IEEE exp and divide
__device__ __forceinline__ float silu_exact(float x) { return x / (1.0f + expf(-x)); }
__device__ __forceinline__ float sigmoid_exact(float x) { return 1.0f / (1.0f + expf(-x)); }

// ---------------------------------------------------------------------------
// GEMM on v_mfma_f32_16x16x4_f32 (lane l holds A[l % 16][l / 16] and
// B[l / 16][l % 16]; accumulator element r of lane l is C[(l / 16) * 4 + r][l % 16]).
// K is taken in pieces of 16: lane group q = l / 16 supplies elements 4 q + e
// in step e, so that a lane's share of a row is one 16-byte word.  Every kernel
// below sums the 32-deep slices of K in the same eight blocks, each from zero,
// and then the blocks in order: a row's bits do not depend on how many rows
// there are, which decides the kernel (2,048 x 2,048 x 1,024 67 us as one sum a
// tile, 70 by blocks).
//
// Large products, bound by the matrix rate: 64 x 64 tiles (small enough that
// 1,000 rows against 1,024 columns give every CU one), a wave's 16 rows x 64
// columns, K in 32-deep slices through a ring of kSlots LDS slots filled by
// direct loads.  A slice row is 128 bytes; its 16-byte chunk c is stored at
// chunk c ^ ((row >> 1) & 7), so that the 16 rows of a fragment read hit 16
// distinct bank groups.  One wave per SIMD has nothing to hide its other
// instructions behind but its own MFMAs, so LDS reads and loads are spread
// between them and slot indexes are constants.  1,000 x 7,168 x 1,024 with
// SwiGLU 275 -> 117 us (126 TFLOP/s, inputs in the caches), 1,000 x 1,024 x 3,584
// 399 -> 60 us (123); at 4,096 rows 128 to 139 TFLOP/s of the 150 that MFMAs alone
// reach.
constexpr int kSlots = 4, kSlice = 64 * 32;  // floats of one operand's slice

__device__ __forceinline__ int slices_per_block(int slices) { return (slices + 7) / 8; }

typedef __attribute__((address_space(3))) void lds_void_t;

__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t src, float* lds, uint32_t lane_at,
                                           uint32_t at) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (lds_void_t*)lds, 16, lane_at, at, 0, 0);
}
__device__ __forceinline__ void load_lds4(__amdgpu_buffer_rsrc_t src, float* lds, uint32_t lane_at,
                                          uint32_t at) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (lds_void_t*)lds, 4, lane_at, at, 0, 0);
}

// one output element (or gate / up pair) through the epilogue
__device__ __forceinline__ void gemm_f32_store(int epilogue, float* C, int64_t ldc, const float* R,
                                               int64_t ldr, int64_t row, int col, float v) {
  if (epilogue == KAD_EPI_RESIDUAL) v += R[row * ldr + col];
  C[row * ldc + col] = v;
}

// WIDE: 16-byte loads (16-byte rows, K a multiple of 4), else 4-byte ones.  TAIL:
// the last slice may reach past K.  2,048 x 2,048 x 1,000 180 us as K split over
// waves (below), 69 here, x 1,001 478 and 90.
template <bool WIDE, bool TAIL>
__global__ __launch_bounds__(256) void gemm_f32_tile_kernel(
    const float* __restrict__ A, int64_t lda, const float* __restrict__ Wt, int64_t ldw,
    float* C, int64_t ldc, const float* R, int64_t ldr, int M, int N, int K, int epilogue,
    int mtiles) {
  constexpr int kFl = WIDE ? 4 : 1;          // floats a lane loads
  constexpr int kLPW = 2048 / (64 * kFl * 4);  // loads per wave, operand and slice
  constexpr int kRows = 2 * kFl;             // slice rows a load covers
  __shared__ __attribute__((aligned(1024))) float ring[kSlots][2 * kSlice];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lid = xcd_logical_id(blockIdx.x, gridDim.x);
  const int m0 = (lid % mtiles) * 64, n0 = (lid / mtiles) * 64;
  // a direct load writes 64 x 16 (or 4) bytes in lane order: 8 (2) rows of a
  // slice, and fetches what belongs at its place.  The wave loads row groups
  // wave, wave + 4, ... of each operand; rows past the end repeat the last one
  // (their results are not stored).  Buffer loads take a lane's row as a fixed
  // offset and the slice as a uniform one, which costs no address arithmetic
  // between the MFMAs (offsets below 2 GB: checked by the dispatch), and read
  // nothing past the last row's end: a slice that reaches there is zeroed below.
  auto bounded = [&](const float* p, int64_t ld, int rows) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0,
                                             (int)(((min(rows, 64) - 1) * ld + K) * 4), 0x00020000);
  };
  const __amdgpu_buffer_rsrc_t ab = bounded(A + (int64_t)m0 * lda, lda, M - m0);
  const __amdgpu_buffer_rsrc_t wb = bounded(Wt + (int64_t)n0 * ldw, ldw, N - n0);
  uint32_t ao[kLPW], wo[kLPW];
#pragma unroll
  for (int i = 0; i < kLPW; ++i) {
    const int r = (wave + 4 * i) * kRows + lane / (32 / kFl), at = lane % (32 / kFl) * kFl;
    const int ch = ((at / 4) ^ ((r >> 1) & 7)) * 4 + at % 4;
    ao[i] = (uint32_t)(((int64_t)(min(m0 + r, M - 1) - m0) * lda + ch) * 4);
    wo[i] = (uint32_t)(((int64_t)(min(n0 + r, N - 1) - n0) * ldw + ch) * 4);
  }
  const int KT = (K + 31) / 32;
  // slice t into slot `at`; past the last slice, that one again (never read)
  auto issue = [&](int t, int at) {
    const uint32_t k = (uint32_t)min(t, KT - 1) * 128;
#pragma unroll
    for (int i = 0; i < kLPW; ++i) {
      float* slot = ring[at] + (wave + 4 * i) * kRows * 32;
      if constexpr (WIDE) {
        load_lds16(ab, slot, ao[i], k);
        load_lds16(wb, slot + kSlice, wo[i], k);
      } else {
        load_lds4(ab, slot, ao[i], k);
        load_lds4(wb, slot + kSlice, wo[i], k);
      }
    }
  };
  f32x4_t acc[4], sum[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) acc[g] = sum[g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int fr = lane & 15, fq = lane >> 4, sw = fr >> 1;  // rows differ by multiples of 16
  struct Frags {
    f32x4_t a[2], w[2][4];  // [16-deep piece]
  };
  auto read = [&](Frags& f, int at) {
#pragma unroll
    for (int piece = 0; piece < 2; ++piece) {
      const float* p = ring[at] + fr * 32 + ((piece * 4 + fq) ^ sw) * 4;
      f.a[piece] = *(const f32x4_t*)(p + wave * 16 * 32);
#pragma unroll
      for (int g = 0; g < 4; ++g) f.w[piece][g] = *(const f32x4_t*)(p + kSlice + g * 16 * 32);
    }
  };
  auto mfmas = [&](const Frags& f, int piece) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        acc[g] = mfma16x16x4f32(f.a[piece][e], f.w[piece][g][e], acc[g]);
  };
  // A wave holds slice t in registers when it reaches the barrier between the
  // slice's two halves: after it the slot takes slice t + kSlots, and slice
  // t + 1 (landed by then) is read while the second half multiplies.  The
  // barrier does not wait for the loads still in flight (2 kLPW a slice); the empty
  // asm statements keep LDS accesses on their side of it.
#pragma unroll
  for (int t = 0; t < kSlots; ++t) issue(t, t);
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(2 * kLPW * (kSlots - 1)) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  Frags f[2];
  read(f[0], 0);
  int block_end = slices_per_block(KT);
  // false after the last slice
  auto step = [&](int t, auto slot) -> bool {
    constexpr int at = decltype(slot)::value;
    Frags &cur = f[at & 1], &next = f[(at + 1) & 1];
    if (t == block_end) {
      block_end += slices_per_block(KT);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        sum[g] += acc[g];
        acc[g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
    }
    if constexpr (TAIL) {
      if (t + 1 == KT) {
#pragma unroll
        for (int piece = 0; piece < 2; ++piece)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (t * 32 + piece * 16 + fq * 4 + e >= K) {
              cur.a[piece][e] = 0.f;
#pragma unroll
              for (int g = 0; g < 4; ++g) cur.w[piece][g][e] = 0.f;
            }
      }
    }
    mfmas(cur, 0);
    __builtin_amdgcn_sched_barrier(0);
    if (t + 1 == KT) {
      mfmas(cur, 1);
      return false;
    }
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(2 * kLPW * (kSlots - 2)) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(next, (at + 1) % kSlots);
    issue(t + kSlots, at);
    mfmas(cur, 1);
    // a read (a load) behind each of the first MFMAs
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      if (i < 10) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if (!WIDE || (i >= 10 && i < 14)) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    return true;
  };
  static_assert(kSlots == 4, "one step below for each slot");
  for (int t = 0;; t += kSlots) {
    if (!step(t, std::integral_constant<int, 0>{})) break;
    if (!step(t + 1, std::integral_constant<int, 1>{})) break;
    if (!step(t + 2, std::integral_constant<int, 2>{})) break;
    if (!step(t + 3, std::integral_constant<int, 3>{})) break;
  }
  // no load may land in LDS that is another workgroup's by then
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

#pragma unroll
  for (int g = 0; g < 4; ++g) sum[g] += acc[g];
  const int64_t row0 = m0 + wave * 16 + fq * 4;
  if (epilogue == KAD_EPI_SWIGLU) {
    // the tile's 64 columns are one [gate 32 | up 32] block of W rows
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (row0 + r < M)
          C[(row0 + r) * ldc + n0 / 2 + g * 16 + fr] = silu_exact(sum[g][r]) * sum[g + 2][r];
    return;
  }
#pragma unroll
  for (int g = 0; g < 4; ++g)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (row0 + r < M && n0 + g * 16 + fr < N)
        gemm_f32_store(epilogue, C, ldc, R, ldr, row0 + r, n0 + g * 16 + fr, sum[g][r]);
}

// Short K: 64 x 64 tiles staged through registers and padded LDS rows, few enough
// of both that several workgroups share a CU and hide one another's load, which
// is most of a tile's time, and the output leaves as whole rows (8,192 x 8,192 x
// 32 115 us in the ring tiles, 88 here; x 33 254 and 111).  At most eight
// slices: each is a block.
constexpr int kShortLd = 20, kShortCld = 65;

__global__ __launch_bounds__(256, 6) void gemm_f32_short_kernel(
    const float* __restrict__ A, int64_t lda, const float* __restrict__ Wt, int64_t ldw,
    float* C, int64_t ldc, const float* R, int64_t ldr, int M, int N, int K, int epilogue) {
  // the operands, and then the output
  __shared__ __attribute__((aligned(16))) float as[64 * kShortCld];
  static_assert(2 * kShortLd <= kShortCld, "both operands in the output's place");
  float *ws = as + 64 * kShortLd, *cs = as;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1, fr = lane & 15, fq = lane >> 4;
  const int64_t m0 = (int64_t)blockIdx.y * 64;
  const int n0 = blockIdx.x * 64;
  f32x4_t acc[2][2], sum[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = sum[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < K; k0 += 16) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = tid + u * 256, r = e / 16, c = e % 16;
      as[r * kShortLd + c] = m0 + r < M && k0 + c < K ? A[(m0 + r) * lda + k0 + c] : 0.f;
      ws[r * kShortLd + c] =
          n0 + r < N && k0 + c < K ? Wt[(int64_t)(n0 + r) * ldw + k0 + c] : 0.f;
    }
    __syncthreads();
    f32x4_t a[2], w[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      a[i] = *(const f32x4_t*)&as[(wm * 32 + i * 16 + fr) * kShortLd + fq * 4];
      w[i] = *(const f32x4_t*)&ws[(wn * 32 + i * 16 + fr) * kShortLd + fq * 4];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma16x16x4f32(a[i][e], w[j][e], acc[i][j]);
    if (k0 % 32 || k0 + 16 >= K) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          sum[i][j] += acc[i][j];
          acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        cs[(wm * 32 + i * 16 + fq * 4 + r) * kShortCld + wn * 32 + j * 16 + fr] = sum[i][j][r];
  __syncthreads();
  if (epilogue == KAD_EPI_SWIGLU) {
    for (int e = tid; e < 64 * 32; e += 256) {
      const int r = e / 32, c = e % 32;
      if (m0 + r < M)
        C[(m0 + r) * ldc + n0 / 2 + c] =
            silu_exact(cs[r * kShortCld + c]) * cs[r * kShortCld + 32 + c];
    }
    return;
  }
  for (int e = tid; e < 64 * 64; e += 256) {
    const int r = e / 64, c = e % 64;
    if (m0 + r < M && n0 + c < N)
      gemm_f32_store(epilogue, C, ldc, R, ldr, m0 + r, n0 + c, cs[r * kShortCld + c]);
  }
}

// Products whose 64 x 64 tiles would leave CUs idle: 16 MT rows x 16 columns (SwiGLU: 16 gate and their 16 up
// columns) per workgroup, whose 8 waves take a block of K's slices each,
// operands straight from memory, the next slice loading during the current
// one; the partial sums merge through LDS.  With few rows the weight's bytes
// bound it: 8 rows against 7,168 x 1,024 68 -> 9 us, 1,024 x 3,584 227 -> 13 us.
template <int MT, bool SWIGLU, bool VEC>
__global__ __launch_bounds__(512) void gemm_f32_split_kernel(
    const float* __restrict__ A, int64_t lda, const float* __restrict__ Wt, int64_t ldw,
    float* C, int64_t ldc, const float* R, int64_t ldr, int M, int N, int K, int epilogue,
    int mtiles) {
  constexpr int NG = SWIGLU ? 2 : 1;
  __shared__ __attribute__((aligned(16))) f32x4_t part[8][MT * NG][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lid = xcd_logical_id(blockIdx.x, gridDim.x);
  const int m0 = (lid % mtiles) * 16 * MT, nt = lid / mtiles;
  // SwiGLU: tile nt holds gate rows (nt / 2) * 64 + (nt % 2) * 16 .. of W and
  // the up rows 32 further
  const int n0 = SWIGLU ? (nt >> 1) * 64 + (nt & 1) * 16 : nt * 16;
  const int fr = lane & 15, fq = lane >> 4;
  const float *ap[MT], *wp[NG];
#pragma unroll
  for (int i = 0; i < MT; ++i) ap[i] = A + (int64_t)min(m0 + i * 16 + fr, M - 1) * lda;
#pragma unroll
  for (int g = 0; g < NG; ++g) wp[g] = Wt + (int64_t)min(n0 + g * 32 + fr, N - 1) * ldw;
  auto load4 = [&](const float* p, int k) -> f32x4_t {
    if constexpr (VEC) {  // K a multiple of 4
      return k < K ? *(const f32x4_t*)(p + k) : f32x4_t{0.f, 0.f, 0.f, 0.f};
    } else {
      f32x4_t r;
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = k + e < K ? p[k + e] : 0.f;
      return r;
    }
  };
  f32x4_t acc[MT][NG];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int g = 0; g < NG; ++g) acc[i][g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  f32x4_t a[2][MT], w[2][NG];
  auto load = [&](int u, f32x4_t (&ar)[2][MT], f32x4_t (&wr)[2][NG]) {
#pragma unroll
    for (int piece = 0; piece < 2; ++piece) {
      const int k = u * 32 + piece * 16 + fq * 4;
#pragma unroll
      for (int g = 0; g < NG; ++g) wr[piece][g] = load4(wp[g], k);
#pragma unroll
      for (int i = 0; i < MT; ++i) ar[piece][i] = load4(ap[i], k);
    }
  };
  const int slices = (K + 31) / 32, per = slices_per_block(slices);
  const int end = min(slices, (wave + 1) * per);
  if (wave * per < end) load(wave * per, a, w);
  for (int u = wave * per; u < end; ++u) {
    f32x4_t an[2][MT], wn[2][NG];
    load(u + 1 < end ? u + 1 : u, an, wn);
#pragma unroll
    for (int piece = 0; piece < 2; ++piece)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int g = 0; g < NG; ++g)
            acc[i][g] = mfma16x16x4f32(a[piece][i][e], w[piece][g][e], acc[i][g]);
#pragma unroll
    for (int piece = 0; piece < 2; ++piece) {
#pragma unroll
      for (int i = 0; i < MT; ++i) a[piece][i] = an[piece][i];
#pragma unroll
      for (int g = 0; g < NG; ++g) w[piece][g] = wn[piece][g];
    }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int g = 0; g < NG; ++g) part[wave][i * NG + g][lane] = acc[i][g];
  __syncthreads();
  auto total = [&](int f, int at) {  // element at of fragment f, waves in order
    float v = 0.f;
#pragma unroll
    for (int x = 0; x < 8; ++x) v += ((const float*)part[x][f])[at];
    return v;
  };
  for (int o = tid; o < MT * 256; o += 512) {
    // output (row, column) of the tile, columns fastest
    const int rr = o >> 4, cc = o & 15, i = rr >> 4, r = rr & 15;
    const int at = ((r >> 2) * 16 + cc) * 4 + (r & 3);
    const int64_t row = m0 + rr;
    if (row >= M) continue;
    if constexpr (SWIGLU) {
      C[row * ldc + (nt >> 1) * 32 + (nt & 1) * 16 + cc] =
          silu_exact(total(i * 2, at)) * total(i * 2 + 1, at);
    } else if (n0 + cc < N) {
      gemm_f32_store(epilogue, C, ldc, R, ldr, row, n0 + cc, total(i, at));
    }
  }
}

template <int MT, bool SWIGLU>
void launch_split(bool vec, const float* A, int64_t lda, const float* W, int64_t ldw, float* C,
                  int64_t ldc, const float* R, int64_t ldr, int M, int N, int K, int epilogue,
                  hipStream_t s) {
  const int mtiles = (int)kad_cdiv(M, 16 * MT);
  const dim3 grid((unsigned)(mtiles * kad_cdiv(N, SWIGLU ? 32 : 16)));
  if (vec)
    hipLaunchKernelGGL((gemm_f32_split_kernel<MT, SWIGLU, true>), grid, dim3(512), 0, s, A, lda, W,
                       ldw, C, ldc, R, ldr, M, N, K, epilogue, mtiles);
  else
    hipLaunchKernelGGL((gemm_f32_split_kernel<MT, SWIGLU, false>), grid, dim3(512), 0, s, A, lda, W,
                       ldw, C, ldc, R, ldr, M, N, K, epilogue, mtiles);
}

template <int MT>
void launch_split_epi(bool vec, const float* A, int64_t lda, const float* W, int64_t ldw, float* C,
                      int64_t ldc, const float* R, int64_t ldr, int M, int N, int K, int epilogue,
                      hipStream_t s) {
  if (epilogue == KAD_EPI_SWIGLU)
    launch_split<MT, true>(vec, A, lda, W, ldw, C, ldc, R, ldr, M, N, K, epilogue, s);
  else
    launch_split<MT, false>(vec, A, lda, W, ldw, C, ldc, R, ldr, M, N, K, epilogue, s);
}

// ---------------------------------------------------------------------------
// Row-wise ops: one wave per row (or per head group), elements lane, lane+64, ...
__global__ __launch_bounds__(256) void rmsnorm_f32_kernel(const float* __restrict__ x,
                                                          int64_t ldx, const float* __restrict__ w,
                                                          float w_offset, float* __restrict__ y,
                                                          int64_t ldy, int64_t rows, int D,
                                                          float eps) {
  const int64_t row = (int64_t)blockIdx.x * 4 + threadIdx.x / 64;
  const int lane = threadIdx.x & 63;
  if (row >= rows) return;
  const float* xr = x + row * ldx;
  float ss = 0.f;
  for (int d = lane; d < D; d += 64) ss += xr[d] * xr[d];
  ss = wave_sum(ss);
  const float r = 1.0f / sqrtf(ss / (float)D + eps);
  for (int d = lane; d < D; d += 64) y[row * ldy + d] = (xr[d] * r) * (w_offset + w[d]);
}

__global__ __launch_bounds__(256) void rmsnorm_gated_f32_kernel(
    const float* __restrict__ x, int64_t ldx, const float* __restrict__ z, int64_t ldz,
    const float* __restrict__ w, float* __restrict__ y, int64_t ldy, int64_t groups, int heads,
    int D, float eps) {
  const int64_t g = (int64_t)blockIdx.x * 4 + threadIdx.x / 64;
  const int lane = threadIdx.x & 63;
  if (g >= groups) return;
  const int64_t tok = g / heads;
  const int hh = (int)(g % heads);
  const float* xr = x + tok * ldx + (int64_t)hh * D;
  const float* zr = z + tok * ldz + (int64_t)hh * D;
  float ss = 0.f;
  for (int d = lane; d < D; d += 64) ss += xr[d] * xr[d];
  ss = wave_sum(ss);
  const float r = 1.0f / sqrtf(ss / (float)D + eps);
  for (int d = lane; d < D; d += 64)
    y[tok * ldy + (int64_t)hh * D + d] = (w[d] * (xr[d] * r)) * silu_exact(zr[d]);
}

__global__ __launch_bounds__(256) void gdn_gates_f32_kernel(
    const float* __restrict__ a, int64_t lda, const float* __restrict__ b, int64_t ldb,
    const float* __restrict__ A_log, const float* __restrict__ dt_bias, float* __restrict__ g,
    float* __restrict__ beta, int64_t rows, int HV) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= rows * HV) return;
  const int64_t r = idx / HV;
  const int h = (int)(idx % HV);
  g[idx] = -expf(A_log[h]) * softplus_f(a[r * lda + h] + dt_bias[h]);
  beta[idx] = sigmoid_exact(b[r * ldb + h]);
}

// one wave per (token, head); output layout as kad_qk_norm_rope
__global__ __launch_bounds__(256) void qk_norm_rope_f32_kernel(
    const float* __restrict__ src, int64_t ld_src, int64_t src_head_stride, int heads,
    const float* __restrict__ w, float* __restrict__ dst, int64_t period, int64_t s_b,
    int64_t s_t, int64_t s_h, int64_t rows, int D, int rot, const float* __restrict__ inv_freq,
    int64_t pos0, int64_t pos_period, float eps, int do_norm) {
  const int64_t gw = (int64_t)blockIdx.x * 4 + threadIdx.x / 64;
  const int lane = threadIdx.x & 63;
  if (gw >= rows * heads) return;
  const int64_t tok = gw / heads;
  const int hh = (int)(gw % heads);
  const float* s = src + tok * ld_src + hh * src_head_stride;
  float ss = 0.f;
  for (int d = lane; d < D; d += 64) ss += s[d] * s[d];
  ss = wave_sum(ss);
  const float r = 1.0f / sqrtf(ss / (float)D + eps);
  auto normed = [&](int d) { return do_norm ? (s[d] * r) * (1.0f + w[d]) : s[d]; };
  const int half = rot / 2;
  const float pos = (float)(pos0 + tok % pos_period);
  float* o = dst + (tok / period) * s_b + (tok % period) * s_t + hh * s_h;
  for (int d = lane; d < D; d += 64) {
    float v = normed(d);
    if (d < rot) {
      const float ang = pos * inv_freq[d % half];
      const int pd = d < half ? d + half : d - half;
      const float partner = normed(pd);
      v = v * cosf(ang) + (d < half ? -partner : partner) * sinf(ang);
    }
    o[d] = v;
  }
}

__global__ __launch_bounds__(256) void embedding_f32_kernel(const int64_t* __restrict__ ids,
                                                            const float* __restrict__ table,
                                                            float* __restrict__ out, int64_t rows,
                                                            int D, int64_t vocab) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= rows * D) return;
  const int64_t r = idx / D;
  int64_t id = ids[r];
  id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
  out[idx] = table[id * D + idx % D];
}

__global__ __launch_bounds__(64) void selftest_f32(const float* a, const float* b, float* c) {
  const int l = threadIdx.x;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  // A[16][4]: lane l holds A[l % 16][l / 16]; B[4][16]: lane l holds B[l / 16][l % 16]
  acc = mfma16x16x4f32(a[(l % 16) * 4 + l / 16], b[(l / 16) * 16 + l % 16], acc);
  for (int r = 0; r < 4; ++r) c[((l / 16) * 4 + r) * 16 + (l % 16)] = acc[r];
}

}  // namespace

extern "C" int kad_gemm_f32(const float* A, int64_t lda, const float* W, int64_t ldw, float* C,
                            int64_t ldc, const float* R, int64_t ldr, int M, int N, int K,
                            int epilogue, kad_stream_t stream) {
  KAD_REQUIRE(A && W && C, "null pointer argument");
  KAD_REQUIRE(M > 0 && N > 0 && K > 0, "bad dimensions");
  KAD_REQUIRE(epilogue == KAD_EPI_STORE || epilogue == KAD_EPI_RESIDUAL ||
                  epilogue == KAD_EPI_SWIGLU,
              "unknown epilogue %d", epilogue);
  KAD_REQUIRE(epilogue != KAD_EPI_RESIDUAL || R, "residual epilogue needs R");
  KAD_REQUIRE(epilogue != KAD_EPI_SWIGLU || N % 64 == 0, "SwiGLU needs N %% 64 == 0");
  KAD_REQUIRE(lda >= K && ldw >= K, "row strides too small");
  const int n_out = epilogue == KAD_EPI_SWIGLU ? N / 2 : N;
  KAD_REQUIRE(ldc >= n_out && (epilogue != KAD_EPI_RESIDUAL || ldr >= N), "row strides too small");
  const int64_t tiles = kad_cdiv(M, 64) * kad_cdiv(N, 64);
  KAD_REQUIRE(kad_cdiv(M, 64) < 65536, "too many rows for one launch");
  if (kad_cdiv(M, 16) * kad_cdiv(N, 16) > 0x7fffffff) KAD_UNSUPPORTED("gemm grid too large");
  const bool vec = K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && ((uintptr_t)A % 16) == 0 &&
                   ((uintptr_t)W % 16) == 0;
  hipStream_t s = (hipStream_t)stream;
  // The tile kernel from 72 tiles: at K = 3,584 it takes 60 us however few of
  // its tiles there are (one per CU), the split one 36 us at 64 tiles' worth
  // of rows and columns and 70 us at 80.  At most 32 rows leave half a tile
  // empty: 32 rows against 7,168 x 1,024 are 13 us split, 20 us in tiles.
  // Beyond 2^23 column tiles its workgroups of 512 no longer fit a grid.
  const int64_t cols = kad_cdiv(N, epilogue == KAD_EPI_SWIGLU ? 32 : 16);
  if (((M > 32 && tiles >= 72) || cols >= (1 << 23)) &&
      (lda > ldw ? lda : ldw) * 64 + K < 0x1fffffff) {
    // 8,192 x 8,192: K 96 193 us against 202 in the ring, 128 244 and 226; rows
    // that are not 16-byte ones 129 277 and 388
    if (K <= (vec ? 96 : 256)) {
      hipLaunchKernelGGL(gemm_f32_short_kernel,
                         dim3((unsigned)kad_cdiv(N, 64), (unsigned)kad_cdiv(M, 64)), dim3(256), 0,
                         s, A, lda, W, ldw, C, ldc, R, ldr, M, N, K, epilogue);
      return kad_launch_status("gemm_f32_short_kernel");
    }
#define KAD_TILE(WIDE, TAIL)                                                                    \
  hipLaunchKernelGGL((gemm_f32_tile_kernel<WIDE, TAIL>), dim3((unsigned)tiles), dim3(256), 0, s, \
                     A, lda, W, ldw, C, ldc, R, ldr, M, N, K, epilogue, (int)kad_cdiv(M, 64))
    if (!vec) KAD_TILE(false, true);
    else if (K % 32) KAD_TILE(true, true);
    else KAD_TILE(true, false);
#undef KAD_TILE
    return kad_launch_status("gemm_f32_tile_kernel");
  }
  if (kad_cdiv(M, 64) * cols >= 256)
    launch_split_epi<4>(vec, A, lda, W, ldw, C, ldc, R, ldr, M, N, K, epilogue, s);
  else if (M > 16 && kad_cdiv(M, 32) * cols >= 64)
    launch_split_epi<2>(vec, A, lda, W, ldw, C, ldc, R, ldr, M, N, K, epilogue, s);
  else
    launch_split_epi<1>(vec, A, lda, W, ldw, C, ldc, R, ldr, M, N, K, epilogue, s);
  return kad_launch_status("gemm_f32_split_kernel");
}

extern "C" int kad_rmsnorm_f32(const float* x, int64_t ldx, const float* w, float w_offset,
                               float* y, int64_t ldy, int64_t rows, int D, float eps,
                               kad_stream_t stream) {
  KAD_REQUIRE(x && w && y, "null pointer argument");
  KAD_REQUIRE(rows > 0 && D > 0 && ldx >= D && ldy >= D, "bad dimensions");
  hipLaunchKernelGGL(rmsnorm_f32_kernel, dim3((unsigned)kad_cdiv(rows, 4)), dim3(256), 0,
                     (hipStream_t)stream, x, ldx, w, w_offset, y, ldy, rows, D, eps);
  return kad_launch_status("rmsnorm_f32_kernel");
}

extern "C" int kad_rmsnorm_gated_f32(const float* x, int64_t ldx, const float* z, int64_t ldz,
                                     const float* w, float* y, int64_t ldy, int64_t rows,
                                     int heads, int D, float eps, kad_stream_t stream) {
  KAD_REQUIRE(x && z && w && y, "null pointer argument");
  KAD_REQUIRE(rows > 0 && heads > 0 && D > 0, "bad dimensions");
  const int64_t groups = rows * heads;
  hipLaunchKernelGGL(rmsnorm_gated_f32_kernel, dim3((unsigned)kad_cdiv(groups, 4)), dim3(256), 0,
                     (hipStream_t)stream, x, ldx, z, ldz, w, y, ldy, groups, heads, D, eps);
  return kad_launch_status("rmsnorm_gated_f32_kernel");
}

extern "C" int kad_gdn_gates_f32(const float* a, int64_t lda, const float* b, int64_t ldb,
                                 const float* A_log, const float* dt_bias, float* g, float* beta,
                                 int64_t rows, int HV, kad_stream_t stream) {
  KAD_REQUIRE(a && b && A_log && dt_bias && g && beta, "null pointer argument");
  KAD_REQUIRE(rows > 0 && HV > 0, "bad dimensions");
  hipLaunchKernelGGL(gdn_gates_f32_kernel, dim3((unsigned)kad_cdiv(rows * HV, 256)), dim3(256), 0,
                     (hipStream_t)stream, a, lda, b, ldb, A_log, dt_bias, g, beta, rows, HV);
  return kad_launch_status("gdn_gates_f32_kernel");
}

extern "C" int kad_qk_norm_rope_f32(const float* src, int64_t ld_src, int64_t src_head_stride,
                                    int heads, const float* w, float* dst, int64_t period,
                                    int64_t s_b, int64_t s_t, int64_t s_h, int64_t rows, int D,
                                    int rot, const float* inv_freq, int64_t pos0,
                                    int64_t pos_period, float eps, int do_norm,
                                    kad_stream_t stream) {
  KAD_REQUIRE(src && dst && inv_freq && (w || !do_norm), "null pointer argument");
  KAD_REQUIRE(rows > 0 && heads > 0 && D > 0, "bad dimensions");
  KAD_REQUIRE(rot >= 0 && rot <= D && rot % 2 == 0, "bad rotary dimension");
  KAD_REQUIRE(period > 0 && pos_period > 0, "bad periods");
  hipLaunchKernelGGL(qk_norm_rope_f32_kernel, dim3((unsigned)kad_cdiv(rows * heads, 4)),
                     dim3(256), 0, (hipStream_t)stream, src, ld_src, src_head_stride, heads, w,
                     dst, period, s_b, s_t, s_h, rows, D, rot, inv_freq, pos0, pos_period, eps,
                     do_norm);
  return kad_launch_status("qk_norm_rope_f32_kernel");
}

extern "C" int kad_embedding_f32(const int64_t* ids, const float* table, float* out,
                                 int64_t rows, int D, int64_t vocab, kad_stream_t stream) {
  KAD_REQUIRE(ids && table && out, "null pointer argument");
  KAD_REQUIRE(rows > 0 && D > 0 && vocab > 0, "bad dimensions");
  hipLaunchKernelGGL(embedding_f32_kernel, dim3((unsigned)kad_cdiv(rows * D, 256)), dim3(256), 0,
                     (hipStream_t)stream, ids, table, out, rows, D, vocab);
  return kad_launch_status("embedding_f32_kernel");
}

extern "C" int kad_selftest_mfma_f32(const float* a, const float* b, float* c,
                                     kad_stream_t stream) {
  KAD_REQUIRE(a && b && c, "null pointer argument");
  hipLaunchKernelGGL(selftest_f32, dim3(1), dim3(64), 0, (hipStream_t)stream, a, b, c);
  return kad_launch_status("selftest_f32");
}
