// Shared by the bf16 GEMM sources: epilogue arithmetic and the entry of the
// small-tile kernel.
#pragma once

#include "kad_common.h"

namespace kad_gemm {

// SiLU of the SwiGLU epilogues: x / (1 + e^-x) with the hardware reciprocal
// (1 ulp) in place of the IEEE divide, which is most of the epilogue's VALU
// work; every tile configuration uses it, so they still agree bit for bit
__device__ __forceinline__ float silu_rcp(float x) {
  return x * __builtin_amdgcn_rcpf(1.0f + __expf(-x));
}

// SwiGLU of two adjacent outputs, bf16(bf16(silu(bf16(g))) * bf16(u)) for
// (g0, u0) in the low half and (g1, u1) in the high half: each bf16
// rounding of the pair is one packed conversion (the same bits as rounding
// each value on its own, with half the conversions and their widenings)
__device__ __forceinline__ uint32_t swiglu2(float g0, float g1, float u0, float u1) {
  const uint32_t gp = pack_bf16x2(g0, g1), up = pack_bf16x2(u0, u1);
  const float ua = __uint_as_float(up << 16), ub = __uint_as_float(up & 0xffff0000u);
  const uint32_t sp =
      pack_bf16x2(silu_rcp(__uint_as_float(gp << 16)), silu_rcp(__uint_as_float(gp & 0xffff0000u)));
  return pack_bf16x2(__uint_as_float(sp << 16) * ua, __uint_as_float(sp & 0xffff0000u) * ub);
}

// tiles of gemm_ring_kernel
enum RingTile { RING_16x16, RING_16x32, RING_32x32, RING_32x64, RING_64x64, RING_128x64 };

// whether the ring kernel takes a product in tiles of this kind
bool ring_ok(RingTile tile, int K, int epilogue);
int launch_ring(RingTile tile, int epilogue, const void* A, int64_t lda, const void* W,
                int64_t ldw, void* C, int64_t ldc, const void* R, int64_t ldr, int M, int N, int K,
                hipStream_t s);

}  // namespace kad_gemm
