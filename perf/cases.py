"""The work that users of this framework have it do, as cases that can be timed.

A case is a dict of plain values.  ``listed`` names the fixed ones, ``draw``
gives more of the same ranges, ``prepare`` makes on the GPU what a program
holds before the call, ``run`` makes the call through the public entry points
and returns its outputs, and ``exact`` computes the same outputs in 64 bits
with plain torch.

Kinds of case:
  gdn        kadllm.ops.gated_delta: beams replayed on shared prefix states
             (decode), or prefix states built from prompts (final=True)
  conv       kadllm.ops.causal_conv1d over the beams' suffixes
  attention  kadllm.ops.prefix_attention, optionally over padded prompts
  select     kadllm.grbeam_search with a caller's own adapter: two levels of
             log-softmax, top-k and history over given logits
  mlp        the norm + SwiGLU block a layer of the model runs (kadllm_amd.layers
             in bf16, kadllm_amd.qwen35_f32 in fp32)
  model      Qwen35GRBeamAdapter: prefill, then the decode levels of a search

Head shapes, hidden sizes and vocabulary are those of the repository's two
model configurations (the 0.8B shape, and the tiny hybrid of the tests).
"""

import math

import torch
import torch.nn.functional as F

import kadllm
from kadllm.adapters import Qwen35GRBeamAdapter, native_model
from kadllm_amd import layers, qwen35_f32
from kadllm_amd.config import qwen35_08b_config, tiny_hybrid_config
from kadllm_amd.qwen35 import pack_mlp
from kadllm_amd.weights import random_state_dict

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
DEVICE = "cuda"
EPS = 1e-6
HIDDEN, INNER = 1024, 3584          # the 0.8B shape's MLP
CHANNELS = 6144                     # its conv channels (q | k | v)
GDN_HEADS, GDN_DIM = 16, 128
Q_HEADS, KV_HEADS, HEAD_DIM = 8, 2, 256
VOCAB = 248320
CONFIGS = {"0.8b": qwen35_08b_config, "tiny": tiny_hybrid_config}


def listed():
    return [
        # one GDN layer's mixer at the full serving batch: 32 requests, 256
        # beams, the third output token replayed with its two predecessors
        {"name": "replay_b32_w256_t3", "kind": "gdn", "dtype": "bf16", "requests": 32,
         "beams": 256, "tokens": 3, "final": False},
        # the same layer in a small service with an ordinary, odd beam width
        {"name": "replay_b8_w50_t2", "kind": "gdn", "dtype": "bf16", "requests": 8,
         "beams": 50, "tokens": 2, "final": False},
        # prefix states of four prompts of a round thousand tokens (a bf16 model's prefill)
        {"name": "prefix_bf16_b4_l1000", "kind": "gdn", "dtype": "bf16", "requests": 4,
         "beams": 1, "tokens": 1000, "final": True},
        # prefix states in full precision: an fp32 model's prefill, odd length
        {"name": "prefix_fp32_b2_l777", "kind": "gdn", "dtype": "fp32", "requests": 2,
         "beams": 1, "tokens": 777, "final": True},
        # the short convolution of that layer, in the operator's [B*W, C, T] layout
        {"name": "conv_b32_w256_t3", "kind": "conv", "dtype": "bf16", "requests": 32,
         "beams": 256, "tokens": 3, "rows": False},
        # one attention layer of the full serving batch, second decode level
        {"name": "attention_b32_w256_l1024", "kind": "attention", "dtype": "bf16",
         "requests": 32, "beams": 256, "tokens": 2, "prefix": 1024, "masked": False},
        # attention of an fp32 model over a batch of padded prompts
        {"name": "attention_fp32_b4_w64_l500", "kind": "attention", "dtype": "fp32",
         "requests": 4, "beams": 64, "tokens": 2, "prefix": 500, "masked": True},
        # selection over the whole vocabulary behind a caller's own model
        {"name": "select_b8_w256", "kind": "select", "dtype": "bf16", "requests": 8,
         "beams": 256, "vocab": VOCAB},
        # one layer's MLP block over a decode level's rows (32 x 256)
        {"name": "mlp_bf16_8192", "kind": "mlp", "dtype": "bf16", "rows": 8192},
        # the block in an fp32 model, over a thousand prompt tokens
        {"name": "mlp_fp32_1000", "kind": "mlp", "dtype": "fp32", "rows": 1000},
        # a whole search's model calls at the full serving batch
        {"name": "model_b32_l1024_w256", "kind": "model", "dtype": "bf16", "shape": "0.8b",
         "requests": 32, "prompt": 1024, "beams": 256, "tokens": 2},
        # a single user's request: one short prompt, ten beams; latency is what counts
        {"name": "model_b1_l100_w10", "kind": "model", "dtype": "bf16", "shape": "0.8b",
         "requests": 1, "prompt": 100, "beams": 10, "tokens": 2},
    ]


def _log_int(rng, lo, hi):
    """A whole number between lo and hi, even over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["gdn", "gdn", "prefix", "conv", "attention", "attention", "select",
                       "mlp", "mlp", "model"])
    if kind == "gdn":
        return {"kind": "gdn", "dtype": rng.choice(["bf16", "bf16", "bf16", "fp32"]),
                "requests": _log_int(rng, 1, 32), "beams": _log_int(rng, 4, 256),
                "tokens": rng.randint(1, 4), "final": False}
    if kind == "prefix":
        dtype = rng.choice(["bf16", "bf16", "fp32"])
        return {"kind": "gdn", "dtype": dtype, "requests": rng.randint(1, 8), "beams": 1,
                "tokens": _log_int(rng, 64, 1500 if dtype == "bf16" else 1000), "final": True}
    if kind == "conv":
        return {"kind": "conv", "dtype": rng.choice(["bf16", "bf16", "fp32"]),
                "requests": _log_int(rng, 1, 32), "beams": _log_int(rng, 4, 256),
                "tokens": rng.randint(1, 4), "rows": rng.random() < 0.5}
    if kind == "attention":
        dtype = rng.choice(["bf16", "bf16", "fp32", "fp16"])
        big = dtype == "bf16"
        return {"kind": "attention", "dtype": dtype,
                "requests": _log_int(rng, 1, 32 if big else 8),
                "beams": _log_int(rng, 4, 256 if big else 64), "tokens": rng.randint(1, 3),
                "prefix": _log_int(rng, 60, 1500 if big else 1000),
                "masked": rng.random() < 0.5}
    if kind == "select":
        return {"kind": "select", "dtype": rng.choice(["bf16", "bf16", "fp32"]),
                "requests": rng.randint(1, 8), "beams": _log_int(rng, 4, 256),
                "vocab": rng.choice([VOCAB, 4096, rng.randint(2000, 100000)])}
    if kind == "mlp":
        dtype = rng.choice(["bf16", "bf16", "fp32"])
        return {"kind": "mlp", "dtype": dtype,
                "rows": _log_int(rng, 8, 32768 if dtype == "bf16" else 4096)}
    dtype = rng.choice(["bf16", "fp32"])
    return {"kind": "model", "dtype": dtype, "shape": "0.8b" if dtype == "bf16" else "tiny",
            "requests": rng.randint(1, 4), "prompt": _log_int(rng, 30, 600),
            "beams": _log_int(rng, 4, 64), "tokens": rng.randint(1, 2)}


# ----------------------------------------------------------------------------
# inputs

def _generator(seed):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    return gen


def prepare(case, seed):
    gen = _generator(seed)
    dt = DTYPES[case["dtype"]]

    def normal(*shape, scale=1.0, dtype=dt):
        return (torch.randn(*shape, generator=gen, device=DEVICE) * scale).to(dtype)

    def uniform(*shape):
        return torch.rand(*shape, generator=gen, device=DEVICE)

    if case["kind"] == "gdn":
        B, W, T, H, D = case["requests"], case["beams"], case["tokens"], GDN_HEADS, GDN_DIM
        # q, k, v leave a SiLU; the gates are -A softplus(a + 1) and sigmoid(b),
        # fp32 and in the model's type, as a layer computes them
        q, k, v = (F.silu(normal(B * W, T, H, D, dtype=torch.float32)).to(dt) for _ in range(3))
        g = -(uniform(H) * 16 + 1e-3) * F.softplus(normal(B * W, T, H, dtype=torch.float32) + 1)
        beta = torch.sigmoid(normal(B * W, T, H, dtype=torch.float32)).to(dt)
        state = normal(B, H, D, D, scale=0.0 if case["final"] else 0.1, dtype=torch.float32)
        return {"case": case, "args": (q, k, v, g, beta, state)}
    if case["kind"] == "conv":
        B, W, T = case["requests"], case["beams"], case["tokens"]
        if case["rows"]:  # channels of a projection's rows
            x = normal(B * W, T, CHANNELS).transpose(1, 2)
        else:
            x = normal(B * W, CHANNELS, T)
        weight = (uniform(CHANNELS, 4) - 0.5).to(dt)
        return {"case": case, "args": (x, normal(B, CHANNELS, 4), weight)}
    if case["kind"] == "attention":
        B, W, T, L = case["requests"], case["beams"], case["tokens"], case["prefix"]
        q = normal(B * W, T, Q_HEADS, HEAD_DIM)
        # prefix K/V as a cache holds them: [B, heads, L, dim], seen as [B, L, heads, dim]
        pk, pv = (normal(B, KV_HEADS, L, HEAD_DIM).transpose(1, 2) for _ in range(2))
        sk, sv = (normal(B * W, T, KV_HEADS, HEAD_DIM) for _ in range(2))
        mask = None
        if case["masked"]:
            length = (uniform(B) * (L / 2) + L / 2).long() + 1
            mask = torch.arange(L, device=DEVICE)[None] < length[:, None]
        return {"case": case, "args": (q, pk, pv, sk, sv), "mask": mask}
    if case["kind"] == "select":
        B, W, V = case["requests"], case["beams"], case["vocab"]
        return {"case": case, "ids": torch.zeros(B, 1, dtype=torch.int64, device=DEVICE),
                "adapter": _GivenLogits(normal(B, V, scale=2.0), normal(B, W, V, scale=2.0))}
    if case["kind"] == "mlp":
        gate, up = (normal(INNER, HIDDEN, scale=0.02) for _ in range(2))
        w_gu, w_down = pack_mlp(gate, up, normal(HIDDEN, INNER, scale=0.02))
        return {"case": case, "x": normal(case["rows"], HIDDEN),
                "norm": normal(HIDDEN, scale=0.1), "w_gu": w_gu, "w_down": w_down}
    cfg = CONFIGS[case["shape"]]()
    sd = _weights(case, cfg, seed)
    B, W, T = case["requests"], case["beams"], case["tokens"]

    def ints(high, *shape):
        return torch.randint(0, high, shape, generator=gen, device=DEVICE)

    ids = ints(cfg.vocab_size, B, case["prompt"])
    # each level's histories: the parents' tokens, then one token more
    histories, parents = [ints(cfg.vocab_size, B, W, 1)], [None]
    for _ in range(T - 1):
        p = ints(W, B, W)
        kept = histories[-1].gather(1, p[:, :, None].expand(-1, -1, histories[-1].shape[2]))
        histories.append(torch.cat((kept, ints(cfg.vocab_size, B, W, 1)), 2))
        parents.append(p)
    return {"case": case, "adapter": Qwen35GRBeamAdapter(*native_model(cfg, sd)), "ids": ids,
            "histories": histories, "parents": parents}


def _weights(case, cfg, seed):
    """Random weights that pass a rounding on as a trained model does and not many
    times larger: unit embeddings, and the projections into the residual stream
    scaled by 1 / sqrt(2 layers).  With the plain draw (0.02 everywhere, tied) the
    logits of the 24-layer bf16 model are 0.12 off their value in 64 bits, so that
    nothing could be told from them; with these 0.012."""
    sd = random_state_dict(cfg, seed=seed, dtype=DTYPES[case["dtype"]], device=DEVICE)
    for name in sd:
        if name.endswith(("out_proj.weight", "o_proj.weight", "down_proj.weight")):
            sd[name] = sd[name] * (2 * len(cfg.layer_types)) ** -0.5
    sd["lm_head.weight"] = sd["embed_tokens.weight"]
    sd["embed_tokens.weight"] = sd["embed_tokens.weight"] * 50
    return sd


class _GivenLogits:
    """A caller's adapter whose model has already computed its logits."""

    def __init__(self, first, second):
        self.first, self.second = first, second

    def prefill(self, input_ids):
        return kadllm.PrefillResult(self.first, None)

    def decode(self, history, state):
        return self.second


# ----------------------------------------------------------------------------
# the calls

@torch.no_grad()
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "gdn":
        return kadllm.gated_delta(*state["args"], beam_width=case["beams"],
                                  return_final_state=case["final"])
    if kind == "conv":
        return kadllm.causal_conv1d(*state["args"], beam_width=case["beams"])
    if kind == "attention":
        return kadllm.prefix_attention(*state["args"], beam_width=case["beams"],
                                       prefix_mask=state["mask"])
    if kind == "select":
        found = kadllm.grbeam_search(state["adapter"], state["ids"], [case["beams"]] * 2)
        return {"tokens": found.tokens, "scores": found.scores, "valid": found.valid}
    if kind == "mlp":
        lib = layers if case["dtype"] == "bf16" else qwen35_f32
        n = lib.rmsnorm(state["x"], state["norm"], EPS)
        h = lib.gemm(n, state["w_gu"], epilogue=lib.EPI_SWIGLU)
        return lib.gemm(h, state["w_down"], epilogue=lib.EPI_RESIDUAL, residual=state["x"])
    adapter = state["adapter"]
    prefix = adapter.prefill(state["ids"])
    outputs, cache = [prefix.logits], None
    for level, (history, parents) in enumerate(zip(state["histories"], state["parents"])):
        if adapter.decode_incremental is not None:
            logits, cache = adapter.decode_incremental(
                history, parents, prefix.state, cache,
                keep_cache=level + 1 < len(state["histories"]))
        else:
            logits = adapter.decode(history, prefix.state)
        outputs.append(logits)
    return outputs


# ----------------------------------------------------------------------------
# what a pass cannot do without

def _params(cfg):
    """(weights of all layers, weights of the head)."""
    H, F_ = cfg.hidden_size, cfg.intermediate_size
    kd = cfg.linear_num_key_heads * cfg.linear_key_head_dim
    vd = cfg.linear_num_value_heads * cfg.linear_value_head_dim
    gdn = H * (2 * kd + 2 * vd + 2 * cfg.linear_num_value_heads) + H * vd
    qd = cfg.num_attention_heads * cfg.head_dim
    attn = H * (2 * qd + 2 * cfg.num_key_value_heads * cfg.head_dim) + H * qd
    total = sum((gdn if kind == "linear_attention" else attn) + 3 * H * F_
                for kind in cfg.layer_types)
    return total, cfg.vocab_size * H


def work(case):
    es = DTYPES[case["dtype"]].itemsize
    kind = case["kind"]
    if kind == "gdn":
        B, T, H, D = case["requests"], case["tokens"], GDN_HEADS, GDN_DIM
        rows = B * case["beams"] * T
        state = B * H * D * D * 4
        # per token and head: state times key, outer product, state times query
        return {"bytes": rows * H * (4 * D * es + 4 + es) + state * (2 if case["final"] else 1),
                "flops": rows * H * 6 * D * D}
    if kind == "conv":
        n = case["requests"] * case["beams"] * case["tokens"] * CHANNELS
        return {"bytes": 2 * n * es + case["requests"] * CHANNELS * 3 * es + CHANNELS * 4 * es,
                "flops": n * 8}
    if kind == "attention":
        B, T, L = case["requests"], case["tokens"], case["prefix"]
        rows = B * case["beams"] * T
        return {"bytes": (2 * rows * Q_HEADS + 2 * rows * KV_HEADS + 2 * B * L * KV_HEADS)
                * HEAD_DIM * es,
                "flops": 4 * rows * Q_HEADS * HEAD_DIM * (L + (T + 1) / 2)}
    if kind == "select":
        n = case["requests"] * (case["beams"] + 1) * case["vocab"]
        return {"bytes": n * es, "flops": 4 * n}
    if kind == "mlp":
        return {"bytes": (2 * case["rows"] * HIDDEN + 3 * HIDDEN * INNER) * es,
                "flops": 6 * case["rows"] * HIDDEN * INNER}
    cfg = CONFIGS[case["shape"]]()
    weights, head = _params(cfg)
    B, L, W, T = case["requests"], case["prompt"], case["beams"], case["tokens"]
    attn = sum(k == "full_attention" for k in cfg.layer_types)
    gdn = len(cfg.layer_types) - attn
    qd = cfg.num_attention_heads * cfg.head_dim
    state = (cfg.linear_num_value_heads * cfg.linear_key_head_dim * cfg.linear_value_head_dim)
    rows = B * L + B * W * T                   # each token through the layers once
    flops = 2 * weights * rows + 2 * head * (B + B * W * T)
    flops += 4 * attn * qd * (B * L * L / 2 + B * W * T * L) + 6 * gdn * state * rows
    return {"bytes": (weights + head) * es * (1 + T) + (B + B * W * T) * cfg.vocab_size * es,
            "flops": flops}


# ----------------------------------------------------------------------------
# tolerances

# Measured on the listed and on drawn cases against 64 bits: bf16 operators are
# 0.0012 to 0.0026 off (their outputs' own rounding), fp32 ones 0.6e-7 to 7e-7,
# the bf16 model's logits 0.012 (largest difference 0.09 of the root mean
# square), the fp32 one's up to 3e-6; the selection's scores 0.7e-7.

def tolerance(case):
    kind, dtype = case["kind"], case["dtype"]
    if kind == "select":
        # scores are fp32 sums of a log-softmax; picks whose scores are that
        # close may come in the other order
        return {"rel": 5e-7, "max": 5e-6, "differ": 0.004}
    if kind == "model":
        return {"rel": 0.03, "max": 0.3} if dtype == "bf16" else {"rel": 1e-5, "max": 3e-4}
    if dtype == "bf16":
        return {"rel": 1e-2, "max": 0.05}
    if dtype == "fp16":
        return {"rel": 1e-3, "max": 1e-2}
    return {"rel": 3e-6, "max": 1e-4}


# ----------------------------------------------------------------------------
# the same in 64 bits

@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "model":
        return _exact_model(case, seed)
    s = prepare(case, seed)
    if kind == "gdn":
        q, k, v, g, beta, state = s["args"]
        B, W = case["requests"], case["beams"]
        parts = [_delta(*(t[b * W:(b + 1) * W].double() for t in (q, k, v, g, beta)),
                        state[b:b + 1].double().expand(W, -1, -1, -1)) for b in range(B)] \
            if not case["final"] else [_delta(*(t.double() for t in (q, k, v, g, beta, state)))]
        out = torch.cat([p[0] for p in parts])
        return (out, parts[0][1]) if case["final"] else out
    if kind == "conv":
        x, taps, weight = s["args"]
        B, W = case["requests"], case["beams"]
        parts = []
        for b in range(B):
            xb = x[b * W:(b + 1) * W].double()
            padded = torch.cat((taps[b:b + 1, :, -3:].double().expand(W, -1, -1), xb), -1)
            parts.append(F.silu(_conv(padded, weight.double())))
        y = torch.cat(parts)
        # laid out as x is
        return y.transpose(1, 2).contiguous().transpose(1, 2) if case["rows"] else y
    if kind == "attention":
        q, pk, pv, sk, sv = s["args"]
        W = case["beams"]
        parts = []
        for b in range(case["requests"]):
            one = slice(b * W, (b + 1) * W)
            parts.append(_attend(*(t.double() for t in (q[one], pk[b], pv[b], sk[one], sv[one])),
                                 None if s["mask"] is None else s["mask"][b]))
        return torch.cat(parts)
    if kind == "select":
        ad, W, V = s["adapter"], case["beams"], case["vocab"]
        scores = []
        for b in range(case["requests"]):
            first = ad.first[b].double().log_softmax(-1).topk(W).values
            rows = [ad.second[b, w].double().log_softmax(-1).topk(W).values + first[w]
                    for w in range(W)]
            scores.append(torch.cat(rows).topk(W).values)
        return {"tokens": None, "scores": torch.stack(scores), "valid": None}
    x, norm = s["x"].double(), s["norm"].double()
    w = s["w_gu"].double().view(-1, 2, 32, HIDDEN)  # gate and up rows alternate by 32
    gate, up = w[:, 0].reshape(-1, HIDDEN), w[:, 1].reshape(-1, HIDDEN)
    n = _norm(x, 1 + norm)
    return x + (F.silu(n @ gate.t()) * (n @ up.t())) @ s["w_down"].double().t()


def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w


def _conv(padded, weight):
    """Width-4 depthwise convolution of [N, C, T + 3] without padding."""
    T = padded.shape[-1] - 3
    return sum(padded[..., i:i + T] * weight[:, i, None] for i in range(4))


def _delta(q, k, v, g, beta, S):
    """The gated delta rule token by token: q, k, v [N, T, H, D], S [N, H, K, V]."""
    q = q * torch.rsqrt(q.square().sum(-1, keepdim=True) + EPS) * q.shape[-1] ** -0.5
    k = k * torch.rsqrt(k.square().sum(-1, keepdim=True) + EPS)
    S, out = S.clone(), torch.empty_like(v)
    for t in range(q.shape[1]):
        S *= g[:, t].exp()[..., None, None]
        u = beta[:, t, :, None] * (v[:, t] - (k[:, t, :, None] @ S).squeeze(-2))
        S += k[:, t, :, :, None] * u[:, :, None]
        out[:, t] = (q[:, t, :, None] @ S).squeeze(-2)
    return out, S


def _attend(q, pk, pv, sk, sv, mask):
    """One request: q, sk, sv [W, T, heads, D]; pk, pv [L, heads, D]; mask [L]."""
    W, T, H, D = q.shape
    L, HK = pk.shape[:2]
    out = torch.empty_like(q)
    for h in range(H):
        j = h * HK // H
        pre = q[:, :, h] @ pk[:, j].t() / math.sqrt(D)
        if mask is not None:
            pre = pre.masked_fill(~mask, -math.inf)
        suf = (q[:, :, h] @ sk[:, :, j].transpose(1, 2).contiguous() / math.sqrt(D)).masked_fill(
            ~torch.ones(T, T, dtype=torch.bool, device=q.device).tril(), -math.inf)
        p = torch.cat((pre, suf), -1).softmax(-1)
        out[:, :, h] = p[..., :L] @ pv[:, j] + p[..., L:] @ sv[:, :, j].contiguous()
    return out


def _exact_model(case, seed):
    """Each level's last logits from whole sequences, prompt and history; None
    where that would take long."""
    if case["requests"] * case["beams"] * case["prompt"] > 20000:
        return None
    s = prepare(case, seed)
    cfg, ids = CONFIGS[case["shape"]](), s["ids"]
    sd = {name: w.double() for name, w in _weights(case, cfg, seed).items()}
    outputs = [_logits(cfg, sd, ids)]
    for history in s["histories"]:
        B, W, T = history.shape
        whole = torch.cat((ids[:, None].expand(-1, W, -1), history), 2).reshape(B * W, -1)
        outputs.append(_logits(cfg, sd, whole).view(B, W, -1))
    return outputs


def _logits(cfg, sd, ids):
    """The hybrid model over [N, P] tokens: logits of the last position."""
    N, P = ids.shape
    x = sd["embed_tokens.weight"][ids]
    for i, kind in enumerate(cfg.layer_types):
        w = {name.split(".", 2)[2]: t for name, t in sd.items() if name.startswith(f"layers.{i}.")}
        n = _norm(x, 1 + w["input_layernorm.weight"])
        mixer = _gdn_layer if kind == "linear_attention" else _attention_layer
        x = x + mixer(cfg, w, n)
        n = _norm(x, 1 + w["post_attention_layernorm.weight"])
        h = F.silu(n @ w["mlp.gate_proj.weight"].t()) * (n @ w["mlp.up_proj.weight"].t())
        x = x + h @ w["mlp.down_proj.weight"].t()
    return _norm(x[:, -1], 1 + sd["norm.weight"]) @ sd["lm_head.weight"].t()


def _gdn_layer(cfg, w, n):
    N, P, _ = n.shape
    H, D = cfg.linear_num_key_heads, cfg.linear_key_head_dim
    qkv = (n @ w["linear_attn.in_proj_qkv.weight"].t()).transpose(1, 2)
    qkv = F.silu(_conv(F.pad(qkv, (3, 0)), w["linear_attn.conv1d.weight"][:, 0])).transpose(1, 2)
    q, k, v = (t.reshape(N, P, H, D) for t in qkv.chunk(3, -1))
    a = n @ w["linear_attn.in_proj_a.weight"].t()
    g = -w["linear_attn.A_log"].exp() * F.softplus(a + w["linear_attn.dt_bias"])
    beta = torch.sigmoid(n @ w["linear_attn.in_proj_b.weight"].t())
    o, _ = _delta(q, k, v, g, beta, q.new_zeros(N, H, D, D))
    z = (n @ w["linear_attn.in_proj_z.weight"].t()).view(N, P, H, D)
    y = _norm(o, w["linear_attn.norm.weight"]) * F.silu(z)
    return y.reshape(N, P, -1) @ w["linear_attn.out_proj.weight"].t()


def _attention_layer(cfg, w, n):
    N, P, _ = n.shape
    H, HK, D = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
    q, gate = (n @ w["self_attn.q_proj.weight"].t()).view(N, P, H, 2 * D).chunk(2, -1)
    k = (n @ w["self_attn.k_proj.weight"].t()).view(N, P, HK, D)
    v = (n @ w["self_attn.v_proj.weight"].t()).view(N, P, HK, D)
    rot = int(D * cfg.partial_rotary_factor)
    freq = cfg.rope_theta ** (-torch.arange(0, rot, 2, device=n.device).double() / rot)
    angle = torch.arange(P, device=n.device).double()[:, None] * freq
    cos, sin = angle.cos().repeat(1, 2)[:, None], angle.sin().repeat(1, 2)[:, None]

    def rotate(x):
        a, rest = x[..., :rot], x[..., rot:]
        turned = torch.cat((-a[..., rot // 2:], a[..., :rot // 2]), -1)
        return torch.cat((a * cos + turned * sin, rest), -1)

    q = rotate(_norm(q, 1 + w["self_attn.q_norm.weight"]))
    k = rotate(_norm(k, 1 + w["self_attn.k_norm.weight"]))
    out = torch.empty_like(q)
    future = torch.ones(P, P, dtype=torch.bool, device=n.device).triu(1)
    for h in range(H):
        j = h * HK // H
        s = q[:, :, h].contiguous() @ k[:, :, j].transpose(1, 2).contiguous() * D ** -0.5
        out[:, :, h] = s.masked_fill(future, -math.inf).softmax(-1) @ v[:, :, j].contiguous()
    y = (out * torch.sigmoid(gate)).reshape(N, P, -1)
    return y @ w["self_attn.o_proj.weight"].t()
