// General-shape kernels (gfx950): any head dimension up to 256, any suffix
// length, fp32 / bf16 / fp16 tensors, fp32 arithmetic.
//
// The specialised kernels (factored suffix replay, chunked GDN, prefix-shared
// MFMA attention) cover the Qwen3.5 shapes: head dims 64/128/256, suffixes of
// a few tokens, bf16.  The reference operators accept any shape and dtype
// (src/kadllm/ops.py:70-163,252-341), and its own toy model runs 8-wide heads
// in fp32 over whole prompts (src/kadllm/adapters/reference.py:56-91).  These
// kernels serve every shape outside the specialised set, with the arithmetic
// of the reference's torch path in fp32: the per-token recurrence of
// ops.py:152-158 and one softmax over the prefix and causal suffix keys
// (equal to the two-partition LSE merge of ops.py:229-249,340).

#include <algorithm>
#include <type_traits>
#include <utility>

#include "kad_common.h"

namespace {

__device__ __forceinline__ void store_from_float(void* p, int64_t i, int dtype, float f) {
  if (dtype == KAD_DTYPE_F32)
    ((float*)p)[i] = f;
  else if (dtype == KAD_DTYPE_BF16)
    ((bf16_t*)p)[i] = f2bf(f);
  else
    ((_Float16*)p)[i] = (_Float16)f;
}

// workgroups of 256 in one launch: a grid holds fewer than 2^32 work-items
constexpr int kMaxBlocks = (1 << 24) - 1;

// 1 / (1 + e^-x) with the IEEE exp and divide (torch.sigmoid in fp32)
__device__ __forceinline__ float sigmoid_exact(float x) { return 1.0f / (1.0f + expf(-x)); }

// ---------------------------------------------------------------------------
// Gated delta recurrence.  The value columns of the state evolve independently under
//   S <- S e^{g_t};  u = beta_t (v_t - S^T k_t);  S <- S + k_t u^T;  o_t = S^T q_t
// A column is held by 16 consecutive lanes (K / 16 values each, in registers
// for all T tokens), a workgroup of 4 waves holds 16 columns of one
// (sequence, value head).  A token is one dependent step, so what bounds the
// kernel is the step's length: both dot products (with k, and with q on the
// state before the update, o_t = e^{g} S^T q + (k.q) u) are reduced together
// on DPP permutes within the 16-lane row, and everything that needs no state
// -- the L2 norms (q / sqrt(sum q^2 + 1e-6) * scale, ops.py:147-148), k.q,
// e^g -- is computed for kTile tokens at a time by all lanes, while the next
// tile's loads are in flight.  16 lanes a column give one wave per SIMD at
// 2 sequences x 16 heads x 128 columns, where one lane a column left 64 waves
// (777 fp32 tokens there: 5,970 -> 144 us, 0.19 us a token).
constexpr int kTile = 16;   // tokens staged at a time, one per 16-lane row
constexpr int kCols = 16;   // state columns per workgroup

template <int CTRL>
__device__ __forceinline__ float dpp_row(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL,
                                                               0xF, 0xF, true));
}
// sum over the 16 lanes of a row, in all of them
__device__ __forceinline__ float row16_sum(float x) {
  x += dpp_row<0xB1>(x);   // quad_perm [1, 0, 3, 2]
  x += dpp_row<0x4E>(x);   // quad_perm [2, 3, 0, 1]
  x += dpp_row<0x141>(x);  // row_half_mirror
  x += dpp_row<0x140>(x);  // row_mirror
  return x;
}

// f(0) .. f(15) with the index a compile-time constant
template <typename F, int... I>
__device__ __forceinline__ void unroll16_at(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <typename F>
__device__ __forceinline__ void unroll16(F&& f) {
  unroll16_at(f, std::make_integer_sequence<int, 16>{});
}

// KV values of a column per lane (K <= 16 KV); lane p of a column owns the
// rows c * 16 VW + p VW + e (VW = min(KV, 4)), so that a row of k or q is read
// from LDS as consecutive 16-byte words.
template <typename TIN, int KV>
__global__ __launch_bounds__(256) void gdn_recurrent_kernel(
    const TIN* __restrict__ q, const TIN* __restrict__ k, const TIN* __restrict__ v,
    int64_t ld_qk, int64_t ld_v, const void* __restrict__ gdecay,
    int gate_dtype, const void* __restrict__ beta, int beta_dtype, int64_t ld_gate,
    const void* __restrict__ init, int state_dtype, int beams_per_state, TIN* __restrict__ out,
    int64_t ld_out, float* __restrict__ final_state, int T, int H, int HV, int K, int V,
    float scale, int nvt, int wide, int first) {
  constexpr int VW = KV < 4 ? KV : 4, NC = KV / VW, KP = 16 * KV;
  constexpr int kQK = kTile * KP;   // floats of a tile's k (or q) rows
  constexpr int kStage = 2 * kQK > KP * (kCols + 1) ? 2 * kQK : KP * (kCols + 1);
  typedef float vec_t __attribute__((ext_vector_type(VW)));
  // two tiles of [k | q] rows; the state passes through the first on its way
  // in and out (coalesced rows of 16 columns)
  __shared__ __attribute__((aligned(16))) float rows[2][kStage];
  __shared__ __attribute__((aligned(16))) float scal[2][kTile][4];  // e^g, beta, k.q
  __shared__ float vs[2][kTile][kCols + 1], os[2][kTile][kCols + 1];
  const int tid = threadIdx.x, p = tid & 15, g16 = tid >> 4;
  const int vt = (int)(blockIdx.x % (unsigned)nvt);
  const int64_t nh = blockIdx.x / (unsigned)nvt;
  const int hv = (int)(nh % HV);
  const int64_t n = first + nh / HV;
  const int h = hv / (HV / H);
  const int v0 = vt * kCols, ncol = min(kCols, V - v0);

  float s[KV];
  const int64_t sbase =
      init ? (((n / beams_per_state) * HV + hv) * (int64_t)K) * V + v0 : 0;
#pragma unroll
  for (int i = 0; i < KV; ++i) s[i] = 0.f;
  if (init) {
    for (int r = g16; r < K; r += 16)
      rows[0][r * (kCols + 1) + p] =
          p < ncol ? load_as_float(init, sbase + (int64_t)r * V + p, state_dtype) : 0.f;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < KV; ++i) {
      const int r = (i / VW) * 16 * VW + p * VW + i % VW;
      if (r < K) s[i] = rows[0][r * (kCols + 1) + g16];
    }
    __syncthreads();
  }

  // this thread's share of a tile: KV elements of token g16's q and k rows,
  // column p of its v row, and its gates (every lane of the row loads them)
  TIN rq[KV], rk[KV], rv;
  float rg, rb;
  const TIN* qh = q + (int64_t)h * K;
  const TIN* kh = k + (int64_t)h * K;
  const TIN* vh = v + (int64_t)hv * V + v0;
  auto fetch = [&](int t0) {
    const int64_t row = n * T + min(t0 + g16, T - 1);  // rows past the end are not used
    if (wide) {
      typedef TIN raw_t __attribute__((ext_vector_type(VW)));
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const raw_t a = *(const raw_t*)(qh + row * ld_qk + c * 16 * VW + p * VW);
        const raw_t b = *(const raw_t*)(kh + row * ld_qk + c * 16 * VW + p * VW);
#pragma unroll
        for (int e = 0; e < VW; ++e) {
          rq[c * VW + e] = a[e];
          rk[c * VW + e] = b[e];
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < KV; ++i) {
        const int r = (i / VW) * 16 * VW + p * VW + i % VW;
        rq[i] = r < K ? qh[row * ld_qk + r] : TIN(0);
        rk[i] = r < K ? kh[row * ld_qk + r] : TIN(0);
      }
    }
    rv = p < ncol ? vh[row * ld_v + p] : TIN(0);
    rg = load_as_float(gdecay, row * ld_gate + hv, gate_dtype);
    rb = load_as_float(beta, row * ld_gate + hv, beta_dtype);
  };
  auto stash = [&](int buf) {
    float fq[KV], fk[KV], sq = 0.f, sk = 0.f;
#pragma unroll
    for (int i = 0; i < KV; ++i) {
      fq[i] = Elem<TIN>::to_f(rq[i]);
      fk[i] = Elem<TIN>::to_f(rk[i]);
      sq += fq[i] * fq[i];
      sk += fk[i] * fk[i];
    }
    const float dq = sqrtf(row16_sum(sq) + 1e-6f), dk = sqrtf(row16_sum(sk) + 1e-6f);
    float kq = 0.f;
#pragma unroll
    for (int i = 0; i < KV; ++i) {
      fq[i] = fq[i] / dq * scale;
      fk[i] = fk[i] / dk;
      kq += fk[i] * fq[i];
    }
    kq = row16_sum(kq);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      vec_t a, b;
#pragma unroll
      for (int e = 0; e < VW; ++e) {
        a[e] = fk[c * VW + e];
        b[e] = fq[c * VW + e];
      }
      const int at = g16 * KP + c * 16 * VW + p * VW;
      *(vec_t*)&rows[buf][at] = a;
      *(vec_t*)&rows[buf][kQK + at] = b;
    }
    vs[buf][g16][p] = Elem<TIN>::to_f(rv);
    if (p == 0) {
      scal[buf][g16][0] = expf(rg);
      scal[buf][g16][1] = rb;
      scal[buf][g16][2] = kq;
    }
  };

  fetch(0);
  stash(0);
  __syncthreads();
  const int ntiles = (T + kTile - 1) / kTile;
  for (int tile = 0; tile < ntiles; ++tile) {
    const int buf = tile & 1, t0 = tile * kTile, nt = min(kTile, T - t0);
    if (tile + 1 < ntiles) fetch(t0 + kTile);
    // lane p of a column's row keeps token p's v and gates; a token's values
    // reach the row's other lanes by a DPP row broadcast
    const float tv = vs[buf][p][g16];
    const float4 tg = *(const float4*)scal[buf][p];
    vec_t kv[NC], qv[NC];
    auto load = [&](int t, vec_t (&kr)[NC], vec_t (&qr)[NC]) {
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int at = t * KP + c * 16 * VW + p * VW;
        kr[c] = *(const vec_t*)&rows[buf][at];
        qr[c] = *(const vec_t*)&rows[buf][kQK + at];
      }
    };
    load(0, kv, qv);
    float ot = 0.f;  // token p's output
    auto step = [&](auto tc) {
      constexpr int t = decltype(tc)::value;
      vec_t kn[NC], qn[NC];
      load(t + 1 < kTile ? t + 1 : t, kn, qn);
      const float decay = dpp_row<0x150 + t>(tg.x), bt = dpp_row<0x150 + t>(tg.y);
      const float kq = dpp_row<0x150 + t>(tg.z), vj = dpp_row<0x150 + t>(tv);
      float dk[2] = {0.f, 0.f}, dq[2] = {0.f, 0.f};
#pragma unroll
      for (int i = 0; i < KV; ++i) {
        dk[i & 1] = fmaf(s[i], kv[i / VW][i % VW], dk[i & 1]);
        dq[i & 1] = fmaf(s[i], qv[i / VW][i % VW], dq[i & 1]);
      }
      const float rk = row16_sum(dk[0] + dk[1]), rq = row16_sum(dq[0] + dq[1]);
      const float u = bt * (vj - decay * rk);
#pragma unroll
      for (int i = 0; i < KV; ++i) s[i] = fmaf(kv[i / VW][i % VW], u, s[i] * decay);
      const float o = fmaf(kq, u, decay * rq);
      ot = p == t ? o : ot;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        kv[c] = kn[c];
        qv[c] = qn[c];
      }
    };
    // whole tiles without a branch between tokens, which would hold the next
    // token's LDS reads back until it
    if (nt == kTile)
      unroll16(step);
    else
      unroll16([&](auto tc) {
        if (decltype(tc)::value < nt) step(tc);
      });
    os[buf][p][g16] = ot;
    if (tile + 1 < ntiles) stash(buf ^ 1);
    __syncthreads();
    if (g16 < nt && p < ncol)
      out[(n * T + t0 + g16) * ld_out + (int64_t)hv * V + v0 + p] =
          Elem<TIN>::from_f(os[buf][g16][p]);
  }
  if (final_state) {
#pragma unroll
    for (int i = 0; i < KV; ++i) {
      const int r = (i / VW) * 16 * VW + p * VW + i % VW;
      rows[0][r * (kCols + 1) + g16] = s[i];
    }
    __syncthreads();
    float* f = final_state + ((n * HV + hv) * (int64_t)K) * V + v0;
    if (p < ncol)
      for (int r = g16; r < K; r += 16) f[(int64_t)r * V + p] = rows[0][r * (kCols + 1) + p];
  }
}

template <typename TIN, int KV>
int launch_recurrent(const void* q, const void* k, const void* v, int64_t ld_qk, int64_t ld_v,
                     const void* g, int gate_dtype, const void* beta, int beta_dtype,
                     int64_t ld_gate, const void* init, int state_dtype, int bps, void* out,
                     int64_t ld_out, float* fin, int N, int T, int H, int HV, int K, int V,
                     float scale, hipStream_t s) {
  const int nvt = (V + kCols - 1) / kCols;
  if ((int64_t)HV * nvt > kMaxBlocks) KAD_UNSUPPORTED("too many heads for one launch");
  // whole vectors of min(KV, 4) elements: full, aligned rows
  constexpr int VW = KV < 4 ? KV : 4;
  const int wide = K == 16 * KV && ld_qk % VW == 0 && ((uintptr_t)q % (VW * sizeof(TIN))) == 0 &&
                   ((uintptr_t)k % (VW * sizeof(TIN))) == 0;
  const int per = kMaxBlocks / (HV * nvt);  // sequences of a launch
  for (int first = 0; first < N; first += std::min(per, N - first)) {
    const int blocks = std::min(per, N - first) * HV * nvt;
    hipLaunchKernelGGL((gdn_recurrent_kernel<TIN, KV>), dim3((unsigned)blocks), dim3(256), 0, s,
                       (const TIN*)q, (const TIN*)k, (const TIN*)v, ld_qk, ld_v, g, gate_dtype,
                       beta, beta_dtype, ld_gate, init, state_dtype, bps, (TIN*)out, ld_out, fin,
                       T, H, HV, K, V, scale, nvt, wide, first);
    if (const int rc = kad_launch_status("gdn_recurrent_kernel")) return rc;
  }
  return KAD_OK;
}

// ---------------------------------------------------------------------------
// Prefix + causal-suffix attention in fp32 on v_mfma_f32_16x16x4_f32.
//
// The rows (beam, token, query head of the key head's group) of one key head
// read the same prefix keys, so a workgroup takes 16 of them as the N
// dimension of S^T = K Q^T and its 4 waves take every fourth step of 16 keys:
// the request's prefix keys, then the suffix.  Suffixes of up to 8 tokens go
// one token a step, its 16 keys the tile's beams (a row sees its own); longer
// ones, whole prompts among them, keep to one beam per tile and go 16 tokens a
// step.  Within either order a row's keys come in steps that do not depend on
// which rows share its tile or on how many tokens follow, nor do its bits.  Each wave folds
// its steps with an online softmax into O^T = V^T P^T -- the accumulator of
// S^T is P^T's operand as it stands -- and the four partial results merge
// through LDS.  Splitting the keys over the waves rather than the rows fills
// the chip with 16-row groups: 4 requests x 2 key heads x 512 rows are 256
// workgroups.  Matrix rate bounds it (a step is 2 x 64 MFMAs of 32 cycles at
// head dim 256, against 32 KB of K and V from L2 that arrive meanwhile: V
// during S, the next K during O); 4 requests x 64 beams x 2 tokens, 500 fp32
// keys: 1,100 us as one wave per row, 38 us here (46 while each step loaded its
// mask bytes, behind every load in flight, and scaled to each new maximum).
//
// Masked prefix keys have weight 0 and their V is not read as a number; a row
// with no visible key gives zeros (ops.py:229-240).  The output is rounded to
// the tensor dtype, then multiplied by the rounded sigmoid of the gate when
// one is given (src/kadllm/adapters/qwen3_5.py:199-201).
//
// A product with weight 0 is not left out of an MFMA, so an infinite or NaN V
// entry that a row must not see would reach it.  Rows whose result is not
// finite are therefore computed again one by one (attention_row), skipping
// the keys of weight 0; their sums then run in another order.
struct AttnArgs {
  const void *q, *pk, *pv, *sk, *sv, *gate;
  const uint8_t* mask;
  void* out;
  int64_t sq_n, sq_t, sq_h;
  int64_t sp_b, sp_l, sp_h;
  int64_t ssk_n, ssk_t, ssk_h, ssv_n, ssv_t, ssv_h;
  int64_t sg_n, sg_t, sg_h;
  int64_t so_n, so_t, so_h;
  int W, Tq, Tk, H, HK, L, D;
  int by_token;      // suffix order, see attention_general_kernel
  int beams;         // beams that share a group of rows: W, or 1
  int rows, tiles;   // rows of a group, and its 16-row tiles
  int first;         // the launch's first tile
  float scale;
};

template <typename TIN>
__device__ __forceinline__ void attention_store(const AttnArgs& a, int64_t n, int t, int h, int d,
                                                float y) {
  y = round_to_dtype(y, Elem<TIN>::code);
  if (a.gate) {
    const float g = Elem<TIN>::to_f(((const TIN*)a.gate)[n * a.sg_n + (int64_t)t * a.sg_t +
                                                         (int64_t)h * a.sg_h + d]);
    y = y * round_to_dtype(sigmoid_exact(g), Elem<TIN>::code);
  }
  ((TIN*)a.out)[n * a.so_n + (int64_t)t * a.so_t + (int64_t)h * a.so_h + d] =
      Elem<TIN>::from_f(y);
}

// one row by one wave: lane j scores key j of a tile of 64, lane l
// accumulates output dims l, l + 64, ...; buf: DMAX + 64 floats of LDS of the
// wave's own
template <typename TIN, int DMAX>
__device__ void attention_row(const AttnArgs& a, float* buf, int64_t n, int t, int h) {
  constexpr int R = DMAX / 64;
  float *qv = buf, *ps = buf + DMAX;
  const int lane = threadIdx.x & 63;
  const int64_t b = n / a.W;
  const int hk = h / (a.H / a.HK);
  const int nkeys = a.L + t + (a.Tk - a.Tq) + 1;
  // LDS of one wave is read and written in program order
  auto fence = [] { asm volatile("" ::: "memory"); };
  fence();
  for (int d = lane; d < a.D; d += 64)
    qv[d] = Elem<TIN>::to_f(
        ((const TIN*)a.q)[n * a.sq_n + (int64_t)t * a.sq_t + (int64_t)h * a.sq_h + d]);
  fence();
  auto krow = [&](int key) {
    return key < a.L ? (const TIN*)a.pk + b * a.sp_b + (int64_t)key * a.sp_l + (int64_t)hk * a.sp_h
                     : (const TIN*)a.sk + n * a.ssk_n + (int64_t)(key - a.L) * a.ssk_t +
                           (int64_t)hk * a.ssk_h;
  };
  auto vrow = [&](int key) {
    return key < a.L ? (const TIN*)a.pv + b * a.sp_b + (int64_t)key * a.sp_l + (int64_t)hk * a.sp_h
                     : (const TIN*)a.sv + n * a.ssv_n + (int64_t)(key - a.L) * a.ssv_t +
                           (int64_t)hk * a.ssv_h;
  };
  float m = -INFINITY, l = 0.f;
  float o[R];
#pragma unroll
  for (int r = 0; r < R; ++r) o[r] = 0.f;
  for (int k0 = 0; k0 < nkeys; k0 += 64) {
    const int key = k0 + lane;
    float sc = -INFINITY;
    if (key < nkeys && !(key < a.L && a.mask && a.mask[b * a.L + key] == 0)) {
      const TIN* kp = krow(key);
      float acc = 0.f;
      for (int d = 0; d < a.D; ++d) acc += qv[d] * Elem<TIN>::to_f(kp[d]);
      sc = acc * a.scale;
    }
    const float mn = fmaxf(m, wave_max(sc));
    if (mn == -INFINITY) continue;  // nothing visible yet (masked keys only)
    const float p = sc == -INFINITY ? 0.f : expf(sc - mn);
    const float alpha = m == -INFINITY ? 0.f : expf(m - mn);
    l = l * alpha + wave_sum(p);
    m = mn;
    fence();
    ps[lane] = p;
    fence();
#pragma unroll
    for (int r = 0; r < R; ++r) o[r] *= alpha;
    const int nk = min(64, nkeys - k0);
    for (int jj = 0; jj < nk; ++jj) {
      const float pj = ps[jj];
      if (pj == 0.f) continue;
      const TIN* vp = vrow(k0 + jj);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int d = lane + 64 * r;
        if (d < a.D) o[r] += pj * Elem<TIN>::to_f(vp[d]);
      }
    }
  }
  const float inv = l > 0.f ? 1.0f / l : (l == 0.f ? 0.f : l);  // a NaN sum stays one
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int d = lane + 64 * r;
    if (d < a.D) attention_store<TIN>(a, n, t, h, d, o[r] * inv);
  }
}

// x combined with lane ^ 16's, as max_xor32
__device__ __forceinline__ float max_xor16(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// FULL: head dim DMAX, every row 4-element aligned (whole-vector loads);
// otherwise elements one by one, zero past the head dim
template <typename TIN, int DMAX, bool FULL>
__global__ __launch_bounds__(256, 1) void attention_general_kernel(AttnArgs a) {
  constexpr int NQ = DMAX / 16;   // 16-dim pieces of a row
  constexpr int NV = DMAX / 64;   // 64-dim pieces
  constexpr int LDO = DMAX + 4;   // LDS row of a partial output
  typedef TIN raw4 __attribute__((ext_vector_type(4)));
  __shared__ __attribute__((aligned(16))) float po[4][16 * LDO];
  __shared__ float pm[4][16], pl[4][16];
  __shared__ int again[16];  // rows whose result is not finite
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c = lane & 15, j = lane >> 4;
  const int G = a.H / a.HK;
  const int lid = a.first + xcd_logical_id(blockIdx.x, gridDim.x);
  const int tile = lid % a.tiles;
  const int hk = (lid / a.tiles) % a.HK;
  const int64_t n0 = (int64_t)(lid / a.tiles / a.HK) * a.beams;  // the group's first beam
  const int64_t b = n0 / a.W;
  const int r0 = tile * 16, r1 = min(r0 + 15, a.rows - 1);
  const int w_lo = r0 / (a.Tq * G), w_hi = r1 / (a.Tq * G);
  // this lane's query row (rows past the end repeat the last one)
  const int row = min(r0 + c, a.rows - 1);
  const int qw = row / (a.Tq * G), qt = row / G % a.Tq;
  const int qpos = qt + (a.Tk - a.Tq);  // its suffix position
  // suffix tokens that some row of the tile sees
  const int nsuf = w_lo == w_hi ? (r1 / G % a.Tq) + (a.Tk - a.Tq) + 1 : a.Tk;
  const int psteps = (a.L + 15) / 16;
  const int steps = psteps + (a.by_token ? nsuf : (nsuf + 15) / 16);

  auto load4 = [&](const TIN* p, int d) -> raw4 {
    if constexpr (FULL) {
      return *(const raw4*)(p + d);
    } else {
      raw4 r;
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = d + e < a.D ? p[d + e] : TIN(0);
      return r;
    }
  };
  // key i of step s; past the end the last one
  auto kv_row = [&](bool value, int s, int i) -> const TIN* {
    if (s < psteps) {
      const int key = min(s * 16 + i, a.L - 1);
      return (const TIN*)(value ? a.pv : a.pk) + b * a.sp_b + (int64_t)key * a.sp_l +
             (int64_t)hk * a.sp_h;
    }
    const int64_t n = n0 + (a.by_token ? min(w_lo + i, w_hi) : w_lo);
    const int64_t t = a.by_token ? s - psteps : min((s - psteps) * 16 + i, nsuf - 1);
    return value ? (const TIN*)a.sv + n * a.ssv_n + t * a.ssv_t + (int64_t)hk * a.ssv_h
                 : (const TIN*)a.sk + n * a.ssk_n + t * a.ssk_t + (int64_t)hk * a.ssk_h;
  };

  // v_mfma_f32_16x16x4_f32: lane l holds A[l%16][l/16] and B[l/16][l%16],
  // accumulator element r of lane l is C[(l/16)*4 + r][l%16].  The dims of a
  // 16-dim piece i meet in the order 16 i + 4 j + e (step e), so that a lane
  // reads its share of a row as 4-element vectors.
  // The 16 query rows come through LDS (where the partial outputs go later), one
  // load of each for the four waves.
  float* qs = po[0];
  {
    const int fr = min(r0 + (tid >> 4), a.rows - 1);
    const TIN* qp = (const TIN*)a.q + (n0 + fr / (a.Tq * G)) * a.sq_n +
                    (int64_t)(fr / G % a.Tq) * a.sq_t + (int64_t)(hk * G + fr % G) * a.sq_h;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int d = 64 * i + (tid & 15) * 4;
      const raw4 r = load4(qp, d);
      *(f32x4*)&qs[(tid >> 4) * LDO + d] = f32x4{Elem<TIN>::to_f(r[0]), Elem<TIN>::to_f(r[1]),
                                                 Elem<TIN>::to_f(r[2]), Elem<TIN>::to_f(r[3])};
    }
  }
  raw4 kf[NQ], vf[4][NV];
  // lane c's key of the step: its mask byte, loaded ahead with K (a load in the
  // step itself would wait for every K and V load issued before it)
  uint8_t mbyte = 1;
  auto load_k = [&](int s) {
    if (a.mask && s < psteps) mbyte = a.mask[b * a.L + min(s * 16 + c, a.L - 1)];
    const TIN* p = kv_row(false, s, c);
#pragma unroll
    for (int i = 0; i < NQ; ++i) kf[i] = load4(p, 16 * i + 4 * j);
  };
  f32x4 o[NV * 4];
#pragma unroll
  for (int i = 0; i < NV * 4; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;  // l: this lane's share of the row's sum

  if (tid < 16) again[tid] = 0;
  if (wave < steps) load_k(wave);
  __syncthreads();
  for (int s = wave; s < steps; s += 4) {
    // V of key 4 j + r, dims 64 i + 4 c + e
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const TIN* p = kv_row(true, s, 4 * j + r);
#pragma unroll
      for (int i = 0; i < NV; ++i) vf[r][i] = load4(p, 64 * i + 4 * c);
    }
    // which of this lane's 4 keys its row sees; hidden: nobody does
    bool seen[4], hidden[4];
    const uint32_t visible =
        (uint32_t)__ballot(s >= psteps || (s * 16 + c < a.L && mbyte != 0)) & 0xffffu;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (s < psteps) {
        seen[r] = (visible >> (4 * j + r)) & 1;
        hidden[r] = !seen[r];
      } else if (a.by_token) {
        const int w = w_lo + 4 * j + r;
        seen[r] = w == qw && s - psteps <= qpos;
        hidden[r] = w > w_hi;
      } else {
        const int t = (s - psteps) * 16 + 4 * j + r;
        seen[r] = t <= qpos;
        hidden[r] = t >= nsuf;
      }
    }
    f32x4 acc[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const f32x4 qf = *(const f32x4*)&qs[c * LDO + 16 * i + 4 * j];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        acc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(Elem<TIN>::to_f(kf[i][e]), qf[e], acc[e], 0,
                                                      0, 0);
    }
    if (s + 4 < steps) load_k(s + 4);
    float sc[4], mt = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float x = ((acc[0][r] + acc[1][r]) + (acc[2][r] + acc[3][r])) * a.scale;
      sc[r] = seen[r] ? x : -INFINITY;
      mt = fmaxf(mt, sc[r]);
    }
    mt = max_xor32(max_xor16(mt));
    // m is the row's reference, not its maximum: a row scales what it has only
    // when a score exceeds m by 16 (weights up to e^16 lose nothing in fp32)
    const bool raise = mt > m + 16.f;  // m = -inf: any score
    if (__any(raise)) {
      const float alpha = raise ? (m == -INFINITY ? 0.f : expf(m - mt)) : 1.f;
      l *= alpha;
#pragma unroll
      for (int i = 0; i < NV * 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[i][r] *= alpha;
      if (raise) m = mt;
    }
    float p[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      p[r] = sc[r] == -INFINITY ? 0.f : expf(sc[r] - m);
      l += p[r];
    }
    if (__any(hidden[0] | hidden[1] | hidden[2] | hidden[3])) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (hidden[r])
#pragma unroll
          for (int i = 0; i < NV; ++i) vf[r][i] = raw4{TIN(0), TIN(0), TIN(0), TIN(0)};
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          o[i * 4 + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(Elem<TIN>::to_f(vf[r][i][e]), p[r],
                                                              o[i * 4 + e], 0, 0, 0);
  }
  __syncthreads();  // the query rows are read
  // o[4 i + e][r] is dim 64 i + 4 (4 j + r) + e of row c
  l = add_xor32(add_xor16(l));
  if (lane < 16) {
    pm[wave][lane] = m;
    pl[wave][lane] = l;
  }
#pragma unroll
  for (int i = 0; i < NV; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *(f32x4*)&po[wave][c * LDO + 64 * i + 16 * j + 4 * r] =
          f32x4{o[4 * i][r], o[4 * i + 1][r], o[4 * i + 2][r], o[4 * i + 3][r]};
  __syncthreads();

  // merge: thread -> row tid / 16, dims 64 i + 4 (tid % 16) + e
  const int mr = tid >> 4, md = (tid & 15) * 4;
  float M = -INFINITY, wgt[4], sum = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) M = fmaxf(M, pm[w][mr]);
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    wgt[w] = pm[w][mr] == -INFINITY ? 0.f : expf(pm[w][mr] - M);
    // a wave that saw only NaN scores has no maximum but a NaN sum
    sum += pl[w][mr] != pl[w][mr] ? pl[w][mr] : pl[w][mr] * wgt[w];
  }
  const float inv = sum > 0.f ? 1.0f / sum : (sum == 0.f ? 0.f : sum);
  const int orow = min(r0 + mr, a.rows - 1);
  const int64_t on = n0 + orow / (a.Tq * G);
  const int ot = orow / G % a.Tq, oh = hk * G + orow % G;
  bool finite = true;
  f32x4 y[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    y[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w) y[i] += *(const f32x4*)&po[w][mr * LDO + 64 * i + md] * wgt[w];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      y[i][e] *= inv;
      finite = finite && fabsf(y[i][e]) < INFINITY;
    }
  }
  if (!finite) again[mr] = 1;
  __syncthreads();  // and every partial output is read
  if (r0 + mr < a.rows && !again[mr])
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (64 * i + md + e < a.D) attention_store<TIN>(a, on, ot, oh, 64 * i + md + e, y[i][e]);
  for (int r = r0 + wave; r <= r1; r += 4)
    if (again[r - r0])
      attention_row<TIN, DMAX>(a, po[wave], n0 + r / (a.Tq * G), r / G % a.Tq, hk * G + r % G);
}

template <typename TIN, int DMAX>
int launch_attention(AttnArgs a, int blocks, hipStream_t s) {
  const int64_t strides[] = {a.sq_n, a.sq_t, a.sq_h, a.sp_b, a.sp_l, a.sp_h, a.ssk_n,
                             a.ssk_t, a.ssk_h, a.ssv_n, a.ssv_t, a.ssv_h};
  bool full = a.D == DMAX;
  for (int64_t x : strides) full = full && x % 4 == 0;
  for (const void* p : {a.q, a.pk, a.pv, a.sk, a.sv})
    full = full && ((uintptr_t)p % (4 * sizeof(TIN))) == 0;
  while (a.first < blocks) {
    const int n = std::min(kMaxBlocks, blocks - a.first);
    if (full)
      hipLaunchKernelGGL((attention_general_kernel<TIN, DMAX, true>), dim3(n), dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL((attention_general_kernel<TIN, DMAX, false>), dim3(n), dim3(256), 0, s, a);
    if (const int rc = kad_launch_status("attention_general_kernel")) return rc;
    a.first += n;
  }
  return KAD_OK;
}

template <typename TIN>
int launch_attention_dim(const AttnArgs& a, int blocks, hipStream_t s) {
  if (a.D <= 64) return launch_attention<TIN, 64>(a, blocks, s);
  if (a.D <= 128) return launch_attention<TIN, 128>(a, blocks, s);
  return launch_attention<TIN, 256>(a, blocks, s);
}

}  // namespace

extern "C" int kad_gdn_recurrent(const void* q, const void* k, const void* v, int64_t ld_qk,
                                 int64_t ld_v, int qkv_dtype, const void* log_decay,
                                 int gate_dtype, const void* beta, int beta_dtype,
                                 int64_t ld_gate, const void* initial_state, int state_dtype,
                                 int beams_per_state, void* out, int64_t ld_out,
                                 float* final_state, int N, int T, int H, int HV, int K, int V,
                                 float scale, kad_stream_t stream) {
  KAD_REQUIRE(q && k && v && log_decay && beta && out, "null pointer argument");
  KAD_REQUIRE(N > 0 && T > 0 && H > 0 && HV > 0 && K > 0 && V > 0 && HV % H == 0,
              "bad dimensions");
  KAD_REQUIRE(!initial_state || (beams_per_state > 0 && N % beams_per_state == 0),
              "beams_per_state must divide N");
  KAD_REQUIRE(ld_qk >= (int64_t)H * K && ld_v >= (int64_t)HV * V && ld_out >= (int64_t)HV * V &&
                  ld_gate >= HV,
              "row strides too small");
  for (int dt : {qkv_dtype, gate_dtype, beta_dtype})
    KAD_REQUIRE(dt == KAD_DTYPE_BF16 || dt == KAD_DTYPE_F16 || dt == KAD_DTYPE_F32,
                "unknown dtype code %d", dt);
  KAD_REQUIRE(!initial_state || state_dtype == KAD_DTYPE_F32 || state_dtype == KAD_DTYPE_BF16 ||
                  state_dtype == KAD_DTYPE_F16,
              "unknown state dtype code %d", state_dtype);
  const int bps = initial_state ? beams_per_state : 1;
  hipStream_t s = (hipStream_t)stream;
#define KAD_REC_T(TIN, KV)                                                                      \
  return launch_recurrent<TIN, KV>(q, k, v, ld_qk, ld_v, log_decay, gate_dtype, beta,         \
                                   beta_dtype, ld_gate, initial_state, state_dtype, bps, out, \
                                   ld_out, final_state, N, T, H, HV, K, V, scale, s);
#define KAD_REC(KV)                                                  \
  if (K <= 16 * KV) {                                                \
    if (qkv_dtype == KAD_DTYPE_F32) KAD_REC_T(float, KV)             \
    if (qkv_dtype == KAD_DTYPE_BF16) KAD_REC_T(bf16_t, KV)           \
    KAD_REC_T(_Float16, KV)                                          \
  }
  KAD_REC(1)
  KAD_REC(2)
  KAD_REC(4)
  KAD_REC(8)
  KAD_REC(16)
#undef KAD_REC_T
#undef KAD_REC
  KAD_UNSUPPORTED("gated delta recurrence supports key dims <= 256, got %d", K);
}

extern "C" int kad_attention_general(
    const void* q, int64_t sq_n, int64_t sq_t, int64_t sq_h, const void* prefix_k,
    const void* prefix_v, int64_t sp_b, int64_t sp_l, int64_t sp_h, const void* suffix_k,
    int64_t ssk_n, int64_t ssk_t, int64_t ssk_h, const void* suffix_v, int64_t ssv_n,
    int64_t ssv_t, int64_t ssv_h, const void* prefix_mask, const void* gate, int64_t sg_n,
    int64_t sg_t, int64_t sg_h, void* out, int64_t so_n, int64_t so_t, int64_t so_h, int B,
    int W, int Tq, int Tk, int H, int HK, int L, int D, int dtype, float scale,
    kad_stream_t stream) {
  KAD_REQUIRE(q && suffix_k && suffix_v && out, "null pointer argument");
  KAD_REQUIRE(L == 0 || (prefix_k && prefix_v), "null prefix K/V with L > 0");
  KAD_REQUIRE(B > 0 && W > 0 && Tq > 0 && Tq <= Tk && H > 0 && HK > 0 && H % HK == 0 &&
                  L >= 0 && D > 0,
              "bad dimensions");
  KAD_REQUIRE(dtype == KAD_DTYPE_BF16 || dtype == KAD_DTYPE_F16 || dtype == KAD_DTYPE_F32,
              "unknown dtype code %d", dtype);
  if (D > 256) KAD_UNSUPPORTED("attention supports head dims <= 256, got %d", D);
  const int64_t rows = (int64_t)B * W * Tq * H;
  if (rows > 0x7fffffffLL) KAD_UNSUPPORTED("too many query rows for one launch");
  // The rows of a request's beams share tiles while their suffixes are short:
  // a suffix token is then a step of its own, of which a row uses one key, so
  // past a few tokens a step of 16 of one beam's tokens is less work.
  const int by_token = Tk <= 8;
  const int beams = by_token ? W : 1;
  const int64_t grows = (int64_t)beams * Tq * (H / HK);
  const int64_t tiles = kad_cdiv(grows, 16);
  const int64_t blocks = (int64_t)B * (W / beams) * HK * tiles;
  if (blocks > 0x7fffffffLL) KAD_UNSUPPORTED("too many query rows for one launch");
  const AttnArgs a{q, prefix_k, prefix_v, suffix_k, suffix_v, gate, (const uint8_t*)prefix_mask,
                   out, sq_n, sq_t, sq_h, sp_b, sp_l, sp_h, ssk_n, ssk_t, ssk_h, ssv_n, ssv_t,
                   ssv_h, sg_n, sg_t, sg_h, so_n, so_t, so_h, W, Tq, Tk, H, HK, L, D, by_token,
                   beams, (int)grows, (int)tiles, 0, scale};
  hipStream_t s = (hipStream_t)stream;
  if (dtype == KAD_DTYPE_F32) return launch_attention_dim<float>(a, (int)blocks, s);
  if (dtype == KAD_DTYPE_BF16) return launch_attention_dim<bf16_t>(a, (int)blocks, s);
  return launch_attention_dim<_Float16>(a, (int)blocks, s);
}
