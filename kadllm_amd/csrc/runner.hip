// A Qwen3.5 model's layers enqueued from C: the call sequences of the runner's
// prefill and incremental decode (kadllm_amd/qwen35.py), which follow
// src/kadllm/adapters/qwen3_5.py:106-235, one foreign call per pass instead of
// one per kernel.
//
// A request of one prompt and ten beams launches 740 kernels of 2 to 10 us;
// building each call's arguments in Python took 8 us, so the host bound the
// search (6.3 ms; 4.8 as one call a pass, 2.9 of them the host).  Nothing is
// computed or allocated here: every
// step is an entry point of this library on the caller's stream, with the same
// arguments, hence bits, as the Python sequence, and every buffer is the
// caller's.

#include "kad_common.h"

namespace {

constexpr int kBf = KAD_DTYPE_BF16, kF32 = KAD_DTYPE_F32;

#define KAD_TRY(call)                    \
  do {                                   \
    if (const int rc = (call)) return rc; \
  } while (0)

uint16_t* at(const void* p, int64_t elements) { return (uint16_t*)const_cast<void*>(p) + elements; }

int check_model(const kad_qwen_model* m) {
  KAD_REQUIRE(m && m->layers && m->n_layers > 0, "null model");
  KAD_REQUIRE(m->hidden > 0 && m->ffn > 0 && m->gdn_cols >= m->conv_dim + m->vd + m->ab_rows,
              "bad model dimensions");
  return KAD_OK;
}

// norm, gate | up with SwiGLU, down with the residual
int mlp(const kad_qwen_model& m, const kad_qwen_layer& l, void* x, void* n, void* h, int rows,
        bool prefetch, kad_stream_t s) {
  const int H = m.hidden, F = m.ffn;
  if (prefetch)
    KAD_TRY(kad_cache_prefetch(l.w_gu, (int64_t)4 * F * H, l.w_down, (int64_t)2 * F * H, s));
  KAD_TRY(kad_rmsnorm(x, H, l.post_norm, 1.f, n, H, rows, H, m.eps, s));
  KAD_TRY(kad_gemm_bf16(n, H, l.w_gu, H, h, F, nullptr, 0, rows, 2 * F, H, KAD_EPI_SWIGLU, s));
  return kad_gemm_bf16(h, F, l.w_down, F, x, H, x, H, rows, H, F, KAD_EPI_RESIDUAL, s);
}

int store(const void* a, int64_t lda, const void* w, void* c, int64_t ldc, int M, int N, int K,
          kad_stream_t s) {
  return kad_gemm_bf16(a, lda, w, K, c, ldc, nullptr, 0, M, N, K, KAD_EPI_STORE, s);
}

}  // namespace

extern "C" int kad_qwen_prefill(const kad_qwen_model* m, const kad_qwen_prefill_args* a,
                                kad_stream_t s) {
  KAD_TRY(check_model(m));
  KAD_REQUIRE(a && a->state0 && a->state1 && a->x && a->n && a->h && a->proj && a->mixed && a->q &&
                  a->g && a->beta && a->chunk_ws,
              "null pointer argument");
  KAD_REQUIRE(a->layers >= 0 && a->layers <= m->n_layers && a->B > 0 && a->L > 0,
              "bad dimensions");
  const int B = a->B, L = a->L, rows = B * L, H = m->hidden, C = m->conv_dim, c = C + m->vd;
  const int cols = m->gdn_cols, HV = m->v_heads, nh = m->q_heads, nkv = m->kv_heads;
  const int hd = m->head_dim;
  for (int i = 0; i < a->layers; ++i) {
    const kad_qwen_layer& l = m->layers[i];
    KAD_TRY(kad_rmsnorm(a->x, H, l.input_norm, 1.f, a->n, H, rows, H, m->eps, s));
    if (l.linear) {
      // the gate projection first, while n is in the caches
      KAD_TRY(store(a->n, H, l.w_ab, at(a->proj, c), cols, rows, m->ab_rows, H, s));
      const void* conv = a->proj;
      int64_t ldc = cols;
      if (a->fuse_conv) {
        KAD_TRY(kad_gemm_bf16_conv(a->n, H, l.w_in, H, a->proj, cols, rows, c, H, C, l.conv_w, L,
                                   a->state0[i], a->conv, a->conv_bytes, s));
      } else {
        KAD_TRY(store(a->n, H, l.w_in, a->proj, cols, rows, c, H, s));
        KAD_TRY(kad_causal_conv_prefill(a->proj, cols, l.conv_w, a->conv, C, a->state0[i], B, L, C,
                                        1, s));
        conv = a->conv;
        ldc = C;
      }
      KAD_TRY(kad_gdn_gates(at(a->proj, c), cols, at(a->proj, c + HV), cols, l.A_log, l.dt_bias,
                            a->g, a->beta, rows, HV, s));
      KAD_TRY(kad_gdn_chunk_gated(conv, at(conv, m->kd), at(conv, 2 * m->kd), ldc, ldc, kBf, a->g,
                                  kF32, a->beta, kBf, HV, nullptr, kF32, 1, a->mixed, m->vd,
                                  (float*)a->state1[i], a->chunk_ws, a->chunk_bytes, B, L,
                                  m->k_heads, HV, m->k_dim, m->v_dim, m->gdn_scale,
                                  at(a->proj, C), cols, l.norm_w, m->eps, s));
      KAD_TRY(kad_gemm_bf16(a->mixed, m->vd, l.w_out, m->vd, a->x, H, a->x, H, rows, H, m->vd,
                            KAD_EPI_RESIDUAL, s));
    } else {
      const int ld = (2 * nh + 2 * nkv) * hd;
      KAD_TRY(store(a->n, H, l.w_qkv, a->proj, ld, rows, ld, H, s));
      KAD_TRY(kad_qk_norm_rope(a->proj, ld, 2 * hd, nh, l.q_norm, a->q, rows, 0, nh * hd, hd, rows,
                               hd, m->rot, m->inv_freq, 0, L, m->eps, 1, s));
      const int64_t sb = (int64_t)nkv * L * hd, sh = (int64_t)L * hd;
      KAD_TRY(kad_qk_norm_rope(at(a->proj, 2 * nh * hd), ld, hd, nkv, l.k_norm, a->state0[i], L, sb,
                               hd, sh, rows, hd, m->rot, m->inv_freq, 0, L, m->eps, 1, s));
      KAD_TRY(kad_scatter_heads(at(a->proj, (2 * nh + nkv) * hd), ld, nkv, hd, a->state1[i], L, sb,
                                hd, sh, rows, s));
      const int64_t qb = (int64_t)L * nh * hd;
      KAD_TRY(kad_attention_prefill(a->q, qb, nh * hd, hd, a->state0[i], a->state1[i], sb, hd, sh,
                                    at(a->proj, hd), (int64_t)L * ld, ld, 2 * hd, a->mixed, qb,
                                    nh * hd, hd, B, L, nh, nkv, hd, m->attn_scale, s));
      KAD_TRY(kad_gemm_bf16(a->mixed, nh * hd, l.w_o, nh * hd, a->x, H, a->x, H, rows, H, nh * hd,
                            KAD_EPI_RESIDUAL, s));
    }
    KAD_TRY(mlp(*m, l, a->x, a->n, a->h, rows, false, s));
  }
  return KAD_OK;
}

extern "C" int kad_qwen_decode_step(const kad_qwen_model* m, const kad_qwen_step_args* a,
                                    kad_stream_t s) {
  KAD_TRY(check_model(m));
  KAD_REQUIRE(a && a->prefix && a->x && a->n && a->h && a->mixed && a->q && a->qkv && a->rows_ws &&
                  a->ab && a->g && a->beta,
              "null pointer argument");
  KAD_REQUIRE(a->B > 0 && a->W > 0 && a->T > 0 && a->T <= 2, "bad dimensions");
  KAD_REQUIRE(a->T == 1 || (a->prev0 && a->prev1 && a->parents && a->Wp > 0),
              "no parent rows for a second token");
  KAD_REQUIRE(a->keep ? a->next0 && a->next1 : a->k_ws && a->v_ws, "null pointer argument");
  const int B = a->B, W = a->W, T = a->T, BW = B * W, H = m->hidden, C = m->conv_dim;
  const int c = C + m->vd, cols = m->gdn_cols, HV = m->v_heads, nab = m->ab_rows;
  const int nh = m->q_heads, nkv = m->kv_heads, hd = m->head_dim;
  const int64_t pos = a->pos + T - 1;
  auto follow = [&](const void* src, int64_t ld_src, void* dst, int64_t ld_dst, int64_t bytes) {
    return kad_gather_beam_rows(src, ld_src, T - 1, dst, ld_dst, T, T - 1, bytes, a->parents, B, W,
                                a->Wp, s);
  };
  for (int i = 0; i < m->n_layers; ++i) {
    const kad_qwen_layer& l = m->layers[i];
    const kad_qwen_prefix& p = a->prefix[i];
    if (a->prefetch && !l.linear)
      KAD_TRY(kad_cache_prefetch(l.w_qkv, (int64_t)(2 * nh + 2 * nkv) * hd * H * 2, nullptr, 0, s));
    KAD_TRY(kad_rmsnorm(a->x, H, l.input_norm, 1.f, a->n, H, BW, H, m->eps, s));
    if (l.linear) {
      if (T == 2 && !a->keep && nab % 8 == 0) {
        // the earlier token's rows in place in the parents' cache: only its
        // gate inputs are gathered, in whole 16-byte pieces
        KAD_TRY(follow(at(a->prev0[i], c), (int64_t)cols * 2, a->ab, nab * 2, nab * 2));
        KAD_TRY(store(a->n, H, l.w_ab, at(a->ab, (T - 1) * nab), T * nab, BW, nab, H, s));
        KAD_TRY(store(a->n, H, l.w_in, a->rows_ws, cols, BW, c, H, s));
        KAD_TRY(kad_gdn_gates(a->ab, nab, at(a->ab, HV), nab, l.A_log, l.dt_bias, a->g, a->beta,
                              (int64_t)BW * T, HV, s));
        KAD_TRY(kad_gdn_suffix_replay_conv_gated_parents(
            a->prev0[i], cols, a->parents, a->Wp, a->rows_ws, cols, p.p0, p.s0, p.s1, p.s2,
            p.history, l.conv_w, a->g, kF32, a->beta, kBf, HV, p.p1, p.dtype, at(a->rows_ws, C),
            cols, l.norm_w, m->eps, a->mixed, m->vd, B, W, T, m->k_heads, HV, m->k_dim, m->v_dim,
            m->gdn_scale, s));
      } else {
        void* rows = a->keep ? a->next0[i] : a->rows_ws;
        if (T > 1)
          KAD_TRY(follow(a->prev0[i], (int64_t)cols * 2, rows, (int64_t)cols * 2,
                         (int64_t)cols * 2));
        void* last = at(rows, (int64_t)(T - 1) * cols);
        KAD_TRY(store(a->n, H, l.w_ab, at(last, c), (int64_t)T * cols, BW, nab, H, s));
        KAD_TRY(store(a->n, H, l.w_in, last, (int64_t)T * cols, BW, c, H, s));
        KAD_TRY(kad_gdn_gates(at(rows, c), cols, at(rows, c + HV), cols, l.A_log, l.dt_bias, a->g,
                              a->beta, (int64_t)BW * T, HV, s));
        KAD_TRY(kad_gdn_suffix_replay_conv_gated(
            rows, cols, p.p0, p.s0, p.s1, p.s2, p.history, l.conv_w, a->g, kF32, a->beta, kBf, HV,
            p.p1, p.dtype, at(rows, C), cols, l.norm_w, m->eps, 1, a->mixed, m->vd, B, W, T,
            m->k_heads, HV, m->k_dim, m->v_dim, m->gdn_scale, s));
      }
      KAD_TRY(kad_gemm_bf16(a->mixed, m->vd, l.w_out, m->vd, a->x, H, a->x, H, BW, H, m->vd,
                            KAD_EPI_RESIDUAL, s));
    } else {
      const int ld = (2 * nh + 2 * nkv) * hd;
      const int64_t row = (int64_t)nkv * hd;
      KAD_TRY(store(a->n, H, l.w_qkv, a->qkv, ld, BW, ld, H, s));
      void* k = a->keep ? a->next0[i] : a->k_ws;
      void* v = a->keep ? a->next1[i] : a->v_ws;
      KAD_REQUIRE(k && v, "null pointer argument");
      if (T > 1) {
        KAD_TRY(follow(a->prev0[i], row * 2, k, row * 2, row * 2));
        KAD_TRY(follow(a->prev1[i], row * 2, v, row * 2, row * 2));
      }
      KAD_TRY(kad_qk_norm_rope(a->qkv, ld, 2 * hd, nh, l.q_norm, a->q, BW, 0, nh * hd, hd, BW, hd,
                               m->rot, m->inv_freq, pos, 1, m->eps, 1, s));
      KAD_TRY(kad_qk_norm_rope(at(a->qkv, 2 * nh * hd), ld, hd, nkv, l.k_norm,
                               at(k, (T - 1) * row), BW, 0, T * row, hd, BW, hd, m->rot,
                               m->inv_freq, pos, 1, m->eps, 1, s));
      KAD_TRY(kad_scatter_heads(at(a->qkv, (2 * nh + nkv) * hd), ld, nkv, hd,
                                at(v, (T - 1) * row), BW, 0, T * row, hd, BW, s));
      KAD_TRY(kad_prefix_attention_decode_ex(
          a->q, nh * hd, nh * hd, hd, p.p0, p.p1, p.s0, p.s1, p.s2, k, T * row, row, hd, v,
          T * row, row, hd, nullptr, at(a->qkv, hd), ld, ld, 2 * hd, a->mixed, nh * hd, nh * hd, hd,
          B, W, 1, T, nh, nkv, p.history, hd, m->attn_scale, s));
      KAD_TRY(kad_gemm_bf16(a->mixed, nh * hd, l.w_o, nh * hd, a->x, H, a->x, H, BW, H, nh * hd,
                            KAD_EPI_RESIDUAL, s));
    }
    KAD_TRY(mlp(*m, l, a->x, a->n, a->h, BW, a->prefetch != 0, s));
  }
  return KAD_OK;
}
