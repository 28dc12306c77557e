// bf16 GEMM for few rows (gfx950): C[M, N] = A[M, K] W[N, K]^T as gemm_bf16.hip,
// in tiles of 16 x 16 to 128 x 64 whose K streams through a ring of LDS slots.
//
// With the rows of one request's decode (tens) or prompt (hundreds) the large
// tiles are 8 or 16 workgroups at N = 1,024, each of which pulls megabytes
// through one CU with one 64-deep slice of K in flight.  Small tiles spread the
// same bytes over the chip, and what bounds a workgroup is then latency: the
// first load, and per slice a barrier and an LDS read.  So the ring holds 4
// (8 for the smallest tile) slices of 64 or 128 of K, filled by direct loads
// issued a whole ring ahead, and a wave holds a slice in registers while the
// next one is read.
//
// K accumulates in ascending 32-deep v_mfma_f32_16x16x32_bf16 steps into one
// accumulator per output, which gives the bits of the kernels of
// gemm_bf16.hip; the epilogues round as theirs.  Measured with weights from
// beyond the caches, us a call, the tile that gemm_bf16.hip picks against the
// one it had: N 1,024, K 3,584: 10 rows 6.6 / 42, 100 rows 8.8 / 62, 400 rows
// 13.3 / 65, 2,000 rows 23 / 66; N 8,192, K 1,024: 10 rows 6 / 19 (5.3 is what
// launching costs there), 100 rows 7.7 / 20.

#include <type_traits>

#include "gemm_common.h"

namespace {

using namespace kad_gemm;

typedef __attribute__((address_space(3))) void lds_void_t;

// BM x BN tiles of WM x WN waves; K in slices of BK, SLOTS of them in LDS
template <int BM_, int BN_, int WM_, int WN_, int BK_, int SLOTS_>
struct Ring {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, NW = WM * WN;
  static constexpr int BK = BK_, SLOTS = SLOTS_;
  static constexpr int NI = BM / WM / 16, NJ = BN / WN / 16;  // 16 x 16 blocks per wave
  static constexpr int Slot = (BM + BN) * BK;
  static constexpr int RPI = 512 / BK;                        // rows per load instruction
  static constexpr int LPW = (BM + BN) / RPI / NW;            // loads per wave and slice
  static_assert(LPW * RPI * NW == BM + BN && BM % RPI == 0, "loads must split evenly");
  static_assert(BK == 64 || BK == 128, "swizzles below");
  static_assert(SLOTS % 2 == 0 && LPW * (SLOTS - 1) < 64, "vmcnt counts to 63");
};

// W row of local row r of column tile nt.  SwiGLU: a wave's blocks are its gate
// blocks and then their up blocks, the packed weight [gate 32 | up 32]; the
// tile's outputs are columns nt * BN / 2 ...
template <int EPI, class RG>
__device__ __forceinline__ int weight_row(int nt, int r) {
  if constexpr (EPI == KAD_EPI_SWIGLU) {
    constexpr int H = RG::NJ * 8;  // outputs per wave
    const int wv = r / (2 * H), in = r % (2 * H);
    const int o = nt * (RG::BN / 2) + wv * H + in % H;
    return (o / 32) * 64 + o % 32 + (in >= H ? 32 : 0);
  } else {
    return nt * RG::BN + r;
  }
}

template <int EPI, class RG>
__global__ __launch_bounds__(64 * RG::NW) void gemm_ring_kernel(
    const bf16_t* __restrict__ A, int64_t lda, const bf16_t* __restrict__ Wt, int64_t ldw,
    bf16_t* C, int64_t ldc, const bf16_t* R, int64_t ldr, int M, int N, int K, int mtiles,
    int ntiles, int group, int vec) {
  constexpr int BK = RG::BK, SLOTS = RG::SLOTS, NI = RG::NI, NJ = RG::NJ, NW = RG::NW;
  constexpr int CPR = BK / 8;  // 16-byte chunks per slice row
  constexpr int STEPS = BK / 32;
  __shared__ __attribute__((aligned(1024))) bf16_t ring[SLOTS][RG::Slot];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / RG::WN, wn = wave % RG::WN;
  const int lid = xcd_logical_id(blockIdx.x, gridDim.x);
  // An XCD's run of tiles walks `group` column tiles a row tile at a time: one,
  // so that the rows of few row tiles share their W, or eight, which keeps the
  // run square where a column tile alone would read most of A into each L2
  // (4,096 x 1,024 x 3,584 in 128x64 tiles: 69.4 us by columns, 43.9 by eights;
  // 3,419 rows 56.0 and 42.6, 2,000 rows 25 and 23.2).
  const int g0 = lid / (group * mtiles) * group, in_group = lid - g0 * mtiles;
  const int gw = min(group, ntiles - g0);
  const int mt = in_group / gw, nt = g0 + in_group % gw;
  const int m0 = mt * RG::BM;

  // Chunk c of slice row r is stored at chunk c ^ swizzle(r), so that the 16
  // rows of a fragment read hit 16 distinct bank groups.  A direct load writes
  // 64 x 16 bytes in lane order, RPI rows; lane l fetches the chunk that
  // belongs at its place.  Rows past M or N read a valid row.
  auto swizzle = [](int r) { return BK == 64 ? (r >> 1) & 7 : r & 15; };
  const bf16_t* src[RG::LPW];
#pragma unroll
  for (int i = 0; i < RG::LPW; ++i) {
    const int g = (wave + i * NW) * RG::RPI, r = g + lane / CPR;
    const int ch = ((lane % CPR) ^ swizzle(r)) * 8;
    src[i] = g < RG::BM ? A + (int64_t)min(m0 + r, M - 1) * lda + ch
                        : Wt + (int64_t)min(weight_row<EPI, RG>(nt, r - RG::BM), N - 1) * ldw + ch;
  }
  const int KT = K / BK;
  // slice t into slot `at`; past the last slice, that one again (never read)
  auto issue = [&](int t, int at) {
    const int k = min(t, KT - 1) * BK;
#pragma unroll
    for (int i = 0; i < RG::LPW; ++i)
      __builtin_amdgcn_global_load_lds(
          (__attribute__((address_space(1))) void*)(src[i] + k),
          (lds_void_t*)(ring[at] + (wave + i * NW) * RG::RPI * BK), 16, 0, 0);
  };

  f32x4 acc[NI][NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int fr = lane & 15, fq = lane >> 4;
  struct Frags {
    bf16x8 a[STEPS][NI], w[STEPS][NJ];
  };
  auto read = [&](Frags& f, int at) {
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const int ch = ((s * 4 + fq) ^ swizzle(fr)) * 8;  // rows differ by multiples of 16
      const bf16_t* p = ring[at] + fr * BK + ch;
#pragma unroll
      for (int i = 0; i < NI; ++i)
        f.a[s][i] = as_bf16x8(*(const u32x4*)(p + (wm * NI + i) * 16 * BK));
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        f.w[s][j] = as_bf16x8(*(const u32x4*)(p + (RG::BM + (wn * NJ + j) * 16) * BK));
    }
  };
  auto mfmas = [&](const Frags& f) {
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = mfma16x16x32(f.w[s][j], f.a[s][i], acc[i][j]);
  };
  // Barrier t: slice t + 1 has landed (LPW loads of each later one may be in
  // flight) and every wave holds slice t in registers, so its slot takes slice
  // t + SLOTS; slice t + 1 is read while slice t multiplies.
#pragma unroll
  for (int t = 0; t < SLOTS; ++t) issue(t, t);
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(RG::LPW * (SLOTS - 1)) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  Frags f[2];
  read(f[0], 0);
  // false after the last slice
  auto step = [&](int t, auto slot) -> bool {
    constexpr int at = decltype(slot)::value;
    Frags &cur = f[at & 1], &next = f[(at + 1) & 1];
    if (t + 1 == KT) {
      mfmas(cur);
      return false;
    }
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(RG::LPW * (SLOTS - 2)) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(next, (at + 1) % SLOTS);
    issue(t + SLOTS, at);
    mfmas(cur);
    __builtin_amdgcn_sched_barrier(0);
    return true;
  };
  static_assert(SLOTS == 4 || SLOTS == 8, "one step below for each slot");
  for (int t = 0;; t += SLOTS) {
    if (!step(t, std::integral_constant<int, 0>{})) break;
    if (!step(t + 1, std::integral_constant<int, 1>{})) break;
    if (!step(t + 2, std::integral_constant<int, 2>{})) break;
    if (!step(t + 3, std::integral_constant<int, 3>{})) break;
    if constexpr (SLOTS == 8) {
      if (!step(t + 4, std::integral_constant<int, 4>{})) break;
      if (!step(t + 5, std::integral_constant<int, 5>{})) break;
      if (!step(t + 6, std::integral_constant<int, 6>{})) break;
      if (!step(t + 7, std::integral_constant<int, 7>{})) break;
    }
  }
  // no load may land in LDS that is another workgroup's by then
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // lane: row fr of a block, columns 4 fq .. +3
  constexpr int NO = EPI == KAD_EPI_SWIGLU ? NJ / 2 : NJ;
  const int n_out = EPI == KAD_EPI_SWIGLU ? N / 2 : N;
  const int col0 = (nt * RG::WN + wn) * NO * 16 + fq * 4;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int64_t row = m0 + (wm * NI + i) * 16 + fr;
    if (row >= M) continue;
#pragma unroll
    for (int j = 0; j < NO; ++j) {
      const int col = col0 + j * 16;
      if (col >= n_out) continue;
      bf16_t* c = C + row * ldc + col;
      const bf16_t* r = R + row * ldr + col;
      u32x2 y;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if constexpr (EPI == KAD_EPI_SWIGLU)
          y[h] = swiglu2(acc[i][j][2 * h], acc[i][j][2 * h + 1], acc[i][j + NO][2 * h],
                         acc[i][j + NO][2 * h + 1]);
        else
          y[h] = pack_bf16x2(acc[i][j][2 * h], acc[i][j][2 * h + 1]);
      }
      if (vec) {
        if constexpr (EPI == KAD_EPI_RESIDUAL) {
          const u32x2 rr = *(const u32x2*)r;
#pragma unroll
          for (int h = 0; h < 2; ++h)
            y[h] = pack_bf16x2(
                __uint_as_float(rr[h] << 16) + __uint_as_float(y[h] << 16),
                __uint_as_float(rr[h] & 0xffff0000u) + __uint_as_float(y[h] & 0xffff0000u));
        }
        *(u32x2*)c = y;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (col + e >= n_out) break;
          float v = bf2f((bf16_t)(y[e / 2] >> (16 * (e & 1))));
          if constexpr (EPI == KAD_EPI_RESIDUAL) v += bf2f(r[e]);
          c[e] = f2bf(v);
        }
      }
    }
  }
}

template <int EPI, class RG>
int launch(const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc,
           const void* R, int64_t ldr, int M, int N, int K, hipStream_t s) {
  const int64_t mtiles = kad_cdiv(M, RG::BM), ntiles = kad_cdiv(N, RG::BN);
  const int64_t blocks = mtiles * ntiles;
  if (blocks > 0x7fffffff) KAD_UNSUPPORTED("gemm grid too large");
  const int n_out = EPI == KAD_EPI_SWIGLU ? N / 2 : N;
  const bool vec = n_out % 4 == 0 && ldc % 4 == 0 && ((uintptr_t)C % 8) == 0 &&
                   (EPI != KAD_EPI_RESIDUAL || (ldr % 4 == 0 && ((uintptr_t)R % 8) == 0));
  hipLaunchKernelGGL((gemm_ring_kernel<EPI, RG>), dim3((unsigned)blocks), dim3(64 * RG::NW), 0, s,
                     (const bf16_t*)A, lda, (const bf16_t*)W, ldw, (bf16_t*)C, ldc,
                     (const bf16_t*)R, ldr, M, N, K, (int)mtiles, (int)ntiles,
                     mtiles > 8 ? 8 : 1, (int)vec);
  return kad_launch_status("gemm_ring_kernel");
}

// a wave's SwiGLU blocks come in gate / up pairs: an even number of them
template <int EPI>
int launch_tile(RingTile tile, const void* A, int64_t lda, const void* W, int64_t ldw, void* C,
                int64_t ldc, const void* R, int64_t ldr, int M, int N, int K, hipStream_t s) {
  constexpr bool kPairs = EPI == KAD_EPI_SWIGLU;
#define KAD_RING(...) \
  return launch<EPI, Ring<__VA_ARGS__>>(A, lda, W, ldw, C, ldc, R, ldr, M, N, K, s)
  switch (tile) {
    case RING_16x16:
      if constexpr (!kPairs) KAD_RING(16, 16, 1, 1, 128, 8);
      break;
    case RING_16x32:
      if constexpr (kPairs) KAD_RING(16, 32, 1, 1, 128, 4);
      else KAD_RING(16, 32, 1, 2, 128, 4);
    case RING_32x32:
      if constexpr (kPairs) KAD_RING(32, 32, 2, 1, 128, 4);
      else KAD_RING(32, 32, 2, 2, 128, 4);
    case RING_32x64: KAD_RING(32, 64, 2, 2, 128, 4);
    case RING_64x64: KAD_RING(64, 64, 2, 2, 64, 4);
    case RING_128x64: KAD_RING(128, 64, 4, 2, 64, 4);
  }
#undef KAD_RING
  KAD_UNSUPPORTED("16x16 tiles have no SwiGLU epilogue");
}

}  // namespace

namespace kad_gemm {

bool ring_ok(RingTile tile, int K, int epilogue) {
  if (tile == RING_16x16 && epilogue == KAD_EPI_SWIGLU) return false;
  return K % (tile >= RING_64x64 ? 64 : 128) == 0;
}

int launch_ring(RingTile tile, int epilogue, const void* A, int64_t lda, const void* W,
                int64_t ldw, void* C, int64_t ldc, const void* R, int64_t ldr, int M, int N, int K,
                hipStream_t s) {
  if (!ring_ok(tile, K, epilogue))
    KAD_UNSUPPORTED("ring tile configurations need K a multiple of 128 (64x64: 64) and, for "
                    "SwiGLU, at least 32 columns");
  if (epilogue == KAD_EPI_SWIGLU)
    return launch_tile<KAD_EPI_SWIGLU>(tile, A, lda, W, ldw, C, ldc, R, ldr, M, N, K, s);
  if (epilogue == KAD_EPI_RESIDUAL)
    return launch_tile<KAD_EPI_RESIDUAL>(tile, A, lda, W, ldw, C, ldc, R, ldr, M, N, K, s);
  return launch_tile<KAD_EPI_STORE>(tile, A, lda, W, ldw, C, ldc, R, ldr, M, N, K, s);
}

}  // namespace kad_gemm
