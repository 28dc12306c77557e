"""Native Qwen3.5 prefill / decode / GRBeam search on the GPU against the oracle.

Tolerance.  A bf16 model's logits are only defined up to bf16 rounding noise,
which compounds through depth: on the 24-layer 0.8B shape the oracle's own
bf16 result differs from the same arithmetic in fp32 by ~12% relative L2.
So logits are judged against the oracle evaluated in fp32 on the same bf16
weights ("truth"): the GPU's relative L2 error to the truth must not exceed
the reference arithmetic's own bf16 error by more than 50% (+0.2% absolute),
and single-layer states must match the bf16 oracle to 1e-2.  Token choices are
checked level by level with teacher forcing: the GPU's selection must equal
the oracle's selection applied to the GPU's own logits (exact).
"""

import numpy as np
import pytest
import torch

from kadllm_amd import grbeam_search
from kadllm_amd.adapters import Qwen35GRBeamAdapter, native_model
from kadllm_amd.config import qwen35_08b_config, tiny_hybrid_config
from kadllm_amd.weights import build_hf_text_model, random_state_dict
from oracle import grbeam_ref
from oracle.qwen35_ref import Qwen35Oracle

pytestmark = pytest.mark.gpu


def rel_l2(a, e):
    a, e = a.detach().float().cpu(), e.detach().float().cpu()
    return ((a - e).norm() / e.norm()).item()


def assert_bf16_parity(actual, oracle_bf16, oracle_fp32, name):
    """GPU error to the fp32 truth within 1.5x the reference's own bf16 error."""
    e_ref = rel_l2(oracle_bf16, oracle_fp32)
    e_gpu = rel_l2(actual, oracle_fp32)
    assert torch.isfinite(actual.float()).all(), f"{name}: non-finite"
    assert e_gpu <= 1.5 * e_ref + 2e-3, f"{name}: GPU rel err {e_gpu:.3e} vs bf16 oracle {e_ref:.3e}"
    return e_gpu, e_ref


def assert_logits_close(actual, expected, name, rel=1e-2, max_frac=6e-2):
    a = actual.detach().float().cpu()
    e = expected.detach().float().cpu()
    assert a.shape == e.shape, (name, a.shape, e.shape)
    assert torch.isfinite(a).all(), f"{name}: non-finite"
    r = ((a - e).norm() / e.norm()).item()
    m = ((a - e).abs().max() / e.abs().max()).item()
    assert r <= rel and m <= max_frac, f"{name}: rel L2 {r:.3e}, max {m:.3e}"
    return r


@pytest.fixture(scope="module")
def tiny(device):
    cfg = tiny_hybrid_config()
    sd = random_state_dict(cfg, seed=0, dtype=torch.bfloat16)
    oracle = Qwen35Oracle(cfg, sd)
    model, head = native_model(cfg, {k: v.to(device) for k, v in sd.items()})
    adapter = Qwen35GRBeamAdapter(model, head)
    adapter.truth = Qwen35Oracle(cfg, {k: v.float() for k, v in sd.items()})
    return cfg, oracle, adapter


def test_tiny_prefill_matches_oracle(device, tiny):
    cfg, oracle, adapter = tiny
    g = torch.Generator().manual_seed(0)
    ids = torch.randint(0, cfg.vocab_size, (2, 128), generator=g)
    res = adapter.prefill(ids.to(device))
    torch.cuda.synchronize()
    ref_logits, ref_state = oracle.prefill(ids)
    assert_logits_close(res.logits, ref_logits, "prefill logits")
    for i, (kind, (a, b), (ra, rb)) in enumerate(zip(cfg.layer_types, res.state.layers,
                                                     ref_state.layers)):
        if kind == "linear_attention":
            assert a.shape == ra.shape and b.shape == rb.shape and b.dtype == torch.float32
            assert_logits_close(a, ra, f"layer {i} conv state", rel=1e-2)
            assert_logits_close(b, rb, f"layer {i} recurrent state", rel=2e-2)
        else:
            assert a.shape == ra.shape, (a.shape, ra.shape)
            assert_logits_close(a, ra, f"layer {i} K", rel=1e-2)
            assert_logits_close(b, rb, f"layer {i} V", rel=1e-2)


@pytest.mark.parametrize("T", [1, 2, 3, 5, 6, 8, 10])
def test_tiny_decode_matches_oracle(device, tiny, T):
    cfg, oracle, adapter = tiny
    g = torch.Generator().manual_seed(T)
    ids = torch.randint(0, cfg.vocab_size, (2, 100), generator=g)
    hist = torch.randint(0, cfg.vocab_size, (2, 8, T), generator=g)
    res = adapter.prefill(ids.to(device))
    prefix_before = [(a.clone(), b.clone()) for a, b in res.state.layers]
    logits = adapter.decode(hist.to(device), res.state)
    torch.cuda.synchronize()
    for (a, b), (a0, b0) in zip(res.state.layers, prefix_before):
        assert torch.equal(a, a0) and torch.equal(b, b0), "decode wrote the prefix"
    _, ref_state = oracle.prefill(ids)
    ref = oracle.decode(hist, ref_state)
    _, truth_state = adapter.truth.prefill(ids)
    truth = adapter.truth.decode(hist, truth_state)
    assert_bf16_parity(logits, ref, truth, f"decode T={T}")


def test_tiny_grbeam_teacher_forced(device, tiny):
    cfg, oracle, adapter = tiny
    g = torch.Generator().manual_seed(11)
    ids = torch.randint(0, cfg.vocab_size, (2, 64), generator=g)
    widths = [8, 8, 8]
    result = grbeam_search(adapter, ids.to(device), widths)
    torch.cuda.synchronize()
    assert result.tokens.shape == (2, 8, 3) and result.valid.all()
    toks = result.tokens.cpu()
    for b in range(2):
        assert len({tuple(s) for s in toks[b].tolist()}) == 8, "beams must be distinct"
    # replay the GPU's own path level by level through the oracle
    pre_logits, state = oracle.prefill(ids)
    gpu_pre = adapter.prefill(ids.to(device))
    assert_logits_close(gpu_pre.logits, pre_logits, "level-0 logits")
    scores = torch.zeros(2, 1)
    history = torch.empty(2, 1, 0, dtype=torch.int64)
    logits = gpu_pre.logits.cpu()[:, None]
    for step, w in enumerate(widths):
        if step:
            logits = adapter.decode(history.to(device), gpu_pre.state).cpu()
            assert_logits_close(logits, oracle.decode(history, state), f"level-{step} logits")
        scores, parents, tokens = grbeam_ref.level_select(logits, scores, w)
        history = torch.cat((history.gather(1, parents[..., None].expand(2, w, step)),
                             tokens[..., None]), -1)
    assert torch.equal(history, toks), "GPU search differs from its own teacher-forced replay"
    assert torch.allclose(result.scores.cpu(), scores, atol=1e-4)


def test_transformers_model_input(device):
    """The adapter accepts the transformers Qwen3_5TextModel + lm_head pair."""
    cfg = tiny_hybrid_config()
    sd = random_state_dict(cfg, seed=1, dtype=torch.bfloat16)
    model, head = build_hf_text_model(cfg, {k: v.to(device) for k, v in sd.items()})
    adapter = Qwen35GRBeamAdapter(model, head, gdn_backend="triton", conv_backend="triton",
                                  attention_backend="flash_attn")
    ids = torch.randint(0, cfg.vocab_size, (1, 40), generator=torch.Generator().manual_seed(2))
    res = adapter.prefill(ids.to(device))
    with torch.no_grad():
        hf = head(model(input_ids=ids.to(device)).last_hidden_state[:, -1])
    torch.cuda.synchronize()
    truth, _ = Qwen35Oracle(cfg, {k: v.float() for k, v in sd.items()}).prefill(ids)
    # transformers' own bf16 forward is the yardstick for bf16 rounding noise
    assert_bf16_parity(res.logits, hf, truth, "prefill vs transformers forward")
    with pytest.raises(TypeError):
        Qwen35GRBeamAdapter(torch.nn.Linear(2, 2), head)


def test_08b_shape_prefill_and_decode(device):
    """The 0.8B-shaped model (24 layers, hd 256 attention, GDN 16x128, vocab
    248320) at a small batch: prefill and a 2-token decode against the oracle."""
    cfg = qwen35_08b_config()
    sd = random_state_dict(cfg, seed=0, dtype=torch.bfloat16, device=device)
    model, head = native_model(cfg, sd)
    adapter = Qwen35GRBeamAdapter(model, head)
    oracle = Qwen35Oracle(cfg, {k: v.cpu() for k, v in sd.items()})
    truth = Qwen35Oracle(cfg, {k: v.cpu().float() for k, v in sd.items()})
    g = torch.Generator().manual_seed(4)
    ids = torch.randint(0, cfg.vocab_size, (2, 40), generator=g)
    hist = torch.randint(0, cfg.vocab_size, (2, 4, 2), generator=g)
    res = adapter.prefill(ids.to(device))
    logits = adapter.decode(hist.to(device), res.state)
    torch.cuda.synchronize()
    ref_logits, ref_state = oracle.prefill(ids)
    truth_logits, truth_state = truth.prefill(ids)
    assert_bf16_parity(res.logits, ref_logits, truth_logits, "0.8B prefill logits")
    assert_bf16_parity(logits, oracle.decode(hist, ref_state), truth.decode(hist, truth_state),
                       "0.8B decode logits")


def test_08b_shape_decode_long_suffix(device):
    """The 0.8B shape with 10-token suffixes, past the specialised kernels'
    8: every GDN layer runs the per-token recurrence (key/value dims 128) and
    every attention layer the general kernel (head dim 256), against the oracle;
    the incremental decode of the same histories agrees within bf16 noise."""
    cfg = qwen35_08b_config()
    sd = random_state_dict(cfg, seed=8, dtype=torch.bfloat16, device=device)
    adapter = Qwen35GRBeamAdapter(*native_model(cfg, sd))
    oracle = Qwen35Oracle(cfg, {k: v.cpu() for k, v in sd.items()})
    truth = Qwen35Oracle(cfg, {k: v.cpu().float() for k, v in sd.items()})
    g = torch.Generator().manual_seed(10)
    ids = torch.randint(0, cfg.vocab_size, (2, 36), generator=g)
    hist = torch.randint(0, cfg.vocab_size, (2, 3, 10), generator=g)
    res = adapter.prefill(ids.to(device))
    logits = adapter.decode(hist.to(device), res.state)
    torch.cuda.synchronize()
    _, ref_state = oracle.prefill(ids)
    _, t_state = truth.prefill(ids)
    ref, exact = oracle.decode(hist, ref_state), truth.decode(hist, t_state)
    assert_bf16_parity(logits, ref, exact, "0.8B decode T=10")
    # the same histories built level by level with the cached suffixes: past
    # 8 tokens both paths run the general kernels, whose bf16 results round
    # differently, so each is held to the fp32 truth
    dev_hist = hist.to(device)
    lg, cache = adapter.decode_incremental(dev_hist[:, :, :1], None, res.state, None)
    parents = torch.arange(3, device=device).expand(2, 3).contiguous()
    for t in range(2, 11):
        lg, cache = adapter.decode_incremental(dev_hist[:, :, :t], parents, res.state, cache)
    torch.cuda.synchronize()
    assert_bf16_parity(lg, ref, exact, "0.8B incremental decode T=10")


def _incremental_matches_stateless(adapter, state, B, widths, V, device, seed):
    """Chain decode_incremental over levels with random parents and tokens and
    compare every level's logits with the stateless decode of the same history."""
    g = torch.Generator().manual_seed(seed)
    history = torch.randint(0, V, (B, widths[0], 1), generator=g).to(device)
    logits, cache = adapter.decode_incremental(history, None, state, None)
    assert torch.equal(logits, adapter.decode(history, state)), "level 1"
    for level, W in enumerate(widths[1:], start=2):
        Wp = history.shape[1]
        parents = torch.randint(0, Wp, (B, W), generator=g).to(device)
        tokens = torch.randint(0, V, (B, W, 1), generator=g).to(device)
        history = torch.cat((history.gather(1, parents[..., None].expand(B, W, level - 1)),
                             tokens), -1)
        logits, cache = adapter.decode_incremental(history, parents, state, cache)
        stateless = adapter.decode(history, state)
        torch.cuda.synchronize()
        assert torch.equal(logits, stateless), f"level {level}: incremental logits differ"


def test_incremental_decode_equals_stateless_tiny(device, tiny):
    """Suffix dedup across levels: exactly the stateless replay's logits, T = 1..7
    (past 4 tokens both run the per-token recurrence and the general attention)."""
    cfg, _, adapter = tiny
    ids = torch.randint(0, cfg.vocab_size, (3, 50), generator=torch.Generator().manual_seed(21))
    res = adapter.prefill(ids.to(device))
    _incremental_matches_stateless(adapter, res.state, 3, [5, 7, 6, 9, 4, 3, 5],
                                   cfg.vocab_size, device, 22)


def test_incremental_decode_with_weight_prefetch_equals_stateless(device, tiny):
    """Levels of 2 x 1024 beams, where decode_step reads the MLP and QKV weights
    into the cache ahead of their GEMMs: still exactly the stateless logits."""
    cfg, _, adapter = tiny
    ids = torch.randint(0, cfg.vocab_size, (2, 40), generator=torch.Generator().manual_seed(31))
    res = adapter.prefill(ids.to(device))
    _incremental_matches_stateless(adapter, res.state, 2, [1024, 1024, 1024],
                                   cfg.vocab_size, device, 32)


def test_last_level_without_cache(device, tiny):
    """keep_cache=False (a search's last level): the same logits, no cache."""
    cfg, _, adapter = tiny
    g = torch.Generator().manual_seed(33)
    ids = torch.randint(0, cfg.vocab_size, (2, 40), generator=g)
    res = adapter.prefill(ids.to(device))
    hist = torch.randint(0, cfg.vocab_size, (2, 6, 2), generator=g).to(device)
    _, cache = adapter.decode_incremental(hist[:, :, :1], None, res.state, None)
    parents = torch.arange(6, device=device).expand(2, 6).contiguous()
    kept, cache2 = adapter.decode_incremental(hist, parents, res.state, cache)
    last, none = adapter.decode_incremental(hist, parents, res.state, cache, keep_cache=False)
    torch.cuda.synchronize()
    assert cache2 is not None and none is None
    assert torch.equal(kept, last)


def test_tiny_grbeam_depth7_teacher_forced(device, tiny):
    """A 7-token search (the depth of the reference's README.md:125 runs; the
    reference has no depth limit, src/kadllm/grbeam.py:75-77): every level's
    logits against the oracle, the selection equal to the oracle's on the GPU's
    own logits."""
    cfg, oracle, adapter = tiny
    g = torch.Generator().manual_seed(17)
    B = 2
    ids = torch.randint(0, cfg.vocab_size, (B, 64), generator=g)
    widths = [6, 6, 5, 6, 4, 5, 6]
    result = grbeam_search(adapter, ids.to(device), widths)
    torch.cuda.synchronize()
    toks = result.tokens.cpu()
    assert toks.shape == (B, 6, 7) and result.valid.all()
    pre_logits, state = oracle.prefill(ids)
    _, t_state = adapter.truth.prefill(ids)
    gpu_pre = adapter.prefill(ids.to(device))
    scores = torch.zeros(B, 1)
    history = torch.empty(B, 1, 0, dtype=torch.int64)
    logits = gpu_pre.logits.cpu()[:, None]
    for step, w in enumerate(widths):
        if step:
            logits = adapter.decode(history.to(device), gpu_pre.state).cpu()
            assert_bf16_parity(logits, oracle.decode(history, state),
                               adapter.truth.decode(history, t_state), f"level-{step} logits")
        scores, parents, tokens = grbeam_ref.level_select(logits, scores, w)
        history = torch.cat((history.gather(1, parents[..., None].expand(B, w, step)),
                             tokens[..., None]), -1)
    assert torch.equal(history, toks), "GPU search differs from its own teacher-forced replay"
    assert torch.allclose(result.scores.cpu(), scores, atol=1e-4)


def test_incremental_decode_equals_stateless_08b(device):
    """The 0.8B shape at 4 x 256 beams, where the stateless and incremental
    projections run with different GEMM tile configurations."""
    cfg = qwen35_08b_config()
    sd = random_state_dict(cfg, seed=3, dtype=torch.bfloat16, device=device)
    adapter = Qwen35GRBeamAdapter(*native_model(cfg, sd))
    ids = torch.randint(0, cfg.vocab_size, (4, 64), generator=torch.Generator().manual_seed(5))
    res = adapter.prefill(ids.to(device))
    _incremental_matches_stateless(adapter, res.state, 4, [256, 256], cfg.vocab_size, device, 6)
    # deeper suffixes (5..7 tokens), where the replay and the attention's
    # suffix fold run their long-suffix instantiations in every layer
    res2 = adapter.prefill(ids[:2].to(device))
    _incremental_matches_stateless(adapter, res2.state, 2, [8, 8, 8, 8, 8, 8, 8],
                                   cfg.vocab_size, device, 7)


def test_search_with_and_without_incremental_decode(device, tiny):
    cfg, _, adapter = tiny

    class Stateless:
        def prefill(self, ids):
            return adapter.prefill(ids)

        def decode(self, history, state):
            return adapter.decode(history, state)

    ids = torch.randint(0, cfg.vocab_size, (2, 33), generator=torch.Generator().manual_seed(8))
    a = grbeam_search(adapter, ids.to(device), [6, 9, 7, 5])
    b = grbeam_search(Stateless(), ids.to(device), [6, 9, 7, 5])
    torch.cuda.synchronize()
    assert torch.equal(a.tokens, b.tokens) and torch.equal(a.scores, b.scores)
    assert torch.equal(a.valid, b.valid)


def test_checkpoint_and_cache_interop(device, tmp_path):
    """from_pretrained on a save_pretrained checkpoint equals the in-memory model;
    a transformers prefill cache, taken as the prefix, decodes like the native
    prefix; and the native prefix continues in the transformers forward."""
    from transformers import Qwen3_5ForCausalLM
    cfg = tiny_hybrid_config()
    sd = random_state_dict(cfg, seed=7, dtype=torch.bfloat16)
    model, head = build_hf_text_model(cfg, sd)
    lm = Qwen3_5ForCausalLM(model.config).eval().to(torch.bfloat16)
    lm.model.load_state_dict(model.state_dict())
    lm.lm_head.weight.data.copy_(head.weight.data)
    lm.save_pretrained(tmp_path)
    a1 = Qwen35GRBeamAdapter.from_pretrained(str(tmp_path), device=device)
    a2 = Qwen35GRBeamAdapter(*native_model(cfg, {k: v.to(device) for k, v in sd.items()}))
    g = torch.Generator().manual_seed(9)
    ids = torch.randint(0, cfg.vocab_size, (2, 48), generator=g).to(device)
    hist = torch.randint(0, cfg.vocab_size, (2, 4, 2), generator=g).to(device)
    r1, r2 = a1.prefill(ids), a2.prefill(ids)
    torch.cuda.synchronize()
    assert torch.equal(r1.logits, r2.logits)
    lm = lm.to(device)
    with torch.no_grad():
        out = lm.model(input_ids=ids, use_cache=True, return_dict=True)
    hf_prefix = a1.prefix_from_cache(out.past_key_values, ids.shape[1])
    native = a1.decode(hist, r1.state)
    via_hf = a1.decode(hist, hf_prefix)
    truth = Qwen35Oracle(cfg, {k: v.float() for k, v in sd.items()})
    _, tstate = truth.prefill(ids.cpu())
    exact = truth.decode(hist.cpu(), tstate)
    assert_bf16_parity(via_hf, native, exact, "decode from a transformers prefix")
    cache = a1.prefix_to_cache(r1.state, lm.config)
    nxt = hist[:, 0, :1]
    with torch.no_grad():
        hf_next = lm(input_ids=nxt, past_key_values=cache, use_cache=True).logits[:, -1]
    ours = a1.decode(nxt[:, None, :], r1.state)[:, 0]
    assert_bf16_parity(hf_next, ours, truth.decode(nxt[:, None, :].cpu(), tstate)[:, 0],
                       "transformers continuing the native prefix")


def _widened_state_dict(cfg, seed, extra):
    """A bf16 state dict whose layer i MLP is ``extra[i]`` units wider, as
    WideTuning's to_dense leaves it (src/kadllm/widetuning.py:96-127)."""
    sd = random_state_dict(cfg, seed=seed, dtype=torch.bfloat16)
    g = torch.Generator().manual_seed(seed + 100)
    for i, n in enumerate(extra):
        p = f"layers.{i}.mlp."
        for name in ("gate_proj", "up_proj"):
            w = sd[p + name + ".weight"]
            add = (torch.randn(n, w.shape[1], generator=g) * 0.02).to(w.dtype)
            sd[p + name + ".weight"] = torch.cat((w, add), 0)
        w = sd[p + "down_proj.weight"]
        add = (torch.randn(w.shape[0], n, generator=g) * 0.02).to(w.dtype)
        sd[p + "down_proj.weight"] = torch.cat((w, add), 1)
    return sd


def test_widened_ffn_layers_match_oracle(device):
    """Per-layer FFN widths that are not multiples of the GEMM tiles (768 + 40,
    + 1, + 0, + 232): prefill and a 2-token decode."""
    cfg = tiny_hybrid_config()
    sd = _widened_state_dict(cfg, 12, [40, 1, 0, 232])
    assert sd["layers.0.mlp.gate_proj.weight"].shape[0] == 808
    oracle = Qwen35Oracle(cfg, sd)
    truth = Qwen35Oracle(cfg, {k: v.float() for k, v in sd.items()})
    adapter = Qwen35GRBeamAdapter(*native_model(cfg, {k: v.to(device) for k, v in sd.items()}))
    g = torch.Generator().manual_seed(13)
    ids = torch.randint(0, cfg.vocab_size, (2, 70), generator=g)
    hist = torch.randint(0, cfg.vocab_size, (2, 6, 2), generator=g)
    res = adapter.prefill(ids.to(device))
    logits = adapter.decode(hist.to(device), res.state)
    torch.cuda.synchronize()
    ref_logits, ref_state = oracle.prefill(ids)
    t_logits, t_state = truth.prefill(ids)
    assert_bf16_parity(res.logits, ref_logits, t_logits, "widened prefill")
    assert_bf16_parity(logits, oracle.decode(hist, ref_state), truth.decode(hist, t_state),
                       "widened decode")


def test_gdn_last_layer_pruned_prefill_and_decode(device):
    """A model whose last layer is a GDN layer: the pruned last layer (its
    output gate, out_proj and MLP on the last position only) in the prefill and
    in a 3-token decode, against the oracle."""
    import dataclasses
    cfg = dataclasses.replace(tiny_hybrid_config(), num_hidden_layers=5,
                              layer_types=("linear_attention", "full_attention",
                                           "linear_attention", "full_attention",
                                           "linear_attention"))
    sd = random_state_dict(cfg, seed=21, dtype=torch.bfloat16)
    oracle = Qwen35Oracle(cfg, sd)
    truth = Qwen35Oracle(cfg, {k: v.float() for k, v in sd.items()})
    adapter = Qwen35GRBeamAdapter(*native_model(cfg, {k: v.to(device) for k, v in sd.items()}))
    g = torch.Generator().manual_seed(22)
    ids = torch.randint(0, cfg.vocab_size, (2, 90), generator=g)
    hist = torch.randint(0, cfg.vocab_size, (2, 5, 3), generator=g)
    res = adapter.prefill(ids.to(device))
    logits = adapter.decode(hist.to(device), res.state)
    torch.cuda.synchronize()
    ref_logits, ref_state = oracle.prefill(ids)
    t_logits, t_state = truth.prefill(ids)
    assert_bf16_parity(res.logits, ref_logits, t_logits, "GDN-last prefill")
    assert_bf16_parity(logits, oracle.decode(hist, ref_state), truth.decode(hist, t_state),
                       "GDN-last decode")


def test_sid_only_head_search(device, tiny):
    """A head that projects only to a subset of token ids (in arbitrary order):
    logits are the oracle's columns for those ids, the softmax runs over the
    subset, and the search returns real token ids, each level equal to the
    oracle's selection on the GPU's own logits."""
    cfg, oracle, full = tiny
    g = torch.Generator().manual_seed(31)
    sid = torch.randperm(cfg.vocab_size, generator=g)[:357]
    sd = random_state_dict(cfg, seed=0, dtype=torch.bfloat16)
    adapter = Qwen35GRBeamAdapter(*native_model(cfg, {k: v.to(device) for k, v in sd.items()}),
                                  head_tokens=sid)
    assert torch.equal(adapter.vocab_ids.cpu(), sid)
    ids = torch.randint(0, cfg.vocab_size, (2, 45), generator=g)
    widths = [16, 12, 9]
    result = grbeam_search(adapter, ids.to(device), widths)
    torch.cuda.synchronize()
    toks = result.tokens.cpu()
    assert toks.shape == (2, 9, 3) and result.valid.all()
    assert torch.isin(toks, sid).all(), "search returned a token outside the head"
    pre_logits, state = oracle.prefill(ids)
    t_logits, t_state = full.truth.prefill(ids)
    gpu_pre = adapter.prefill(ids.to(device))
    assert_bf16_parity(gpu_pre.logits, pre_logits[:, sid], t_logits[:, sid], "SID prefill logits")
    # the same model with the full head: its columns for the subset
    assert_logits_close(gpu_pre.logits, full.prefill(ids.to(device)).logits[:, sid.to(device)],
                        "SID vs full-head columns", rel=2e-3, max_frac=1e-2)
    scores = torch.zeros(2, 1)
    history = torch.empty(2, 1, 0, dtype=torch.int64)
    logits = gpu_pre.logits.cpu()[:, None]
    for step, w in enumerate(widths):
        if step:
            logits = adapter.decode(history.to(device), gpu_pre.state).cpu()
            assert logits.shape == (2, history.shape[1], sid.numel())
            assert_bf16_parity(logits, oracle.decode(history, state)[..., sid],
                               full.truth.decode(history, t_state)[..., sid],
                               f"SID level-{step} logits")
        scores, parents, cols = grbeam_ref.level_select(logits, scores, w)
        history = torch.cat((history.gather(1, parents[..., None].expand(2, w, step)),
                             sid[cols][..., None]), -1)
    assert torch.equal(history, toks), "GPU search differs from its own teacher-forced replay"
    assert torch.allclose(result.scores.cpu(), scores, atol=1e-4)
    with pytest.raises(ValueError):
        Qwen35GRBeamAdapter(*native_model(cfg, {k: v.to(device) for k, v in sd.items()}),
                            head_tokens=[cfg.vocab_size])


def test_out_of_range_token_ids_raise(device, tiny):
    """Token ids outside the vocabulary raise IndexError in prefill, decode and
    the incremental decode, as torch's embedding does.  The check is read back
    after the model's kernels are enqueued; those kernels clamp the ids, so
    they stay inside the embedding table."""
    cfg, _, adapter = tiny
    V = cfg.vocab_size
    ids = torch.randint(0, V, (2, 20), generator=torch.Generator().manual_seed(3)).to(device)
    bad = ids.clone()
    bad[1, 7] = V
    with pytest.raises(IndexError, match="index out of range"):
        adapter.prefill(bad)
    bad[1, 7] = -1
    with pytest.raises(IndexError, match="index out of range"):
        adapter.prefill(bad)
    res = adapter.prefill(ids)
    hist = torch.randint(0, V, (2, 3, 2), generator=torch.Generator().manual_seed(4)).to(device)
    hist[0, 2, 1] = V + 5
    with pytest.raises(IndexError, match="index out of range"):
        adapter.decode(hist, res.state)
    with pytest.raises(IndexError, match="index out of range"):
        adapter.decode_incremental(hist[:, :, 1:], None, res.state, None)
    hist[0, 2, 1] = V - 1   # the largest valid id is accepted
    assert adapter.decode(hist, res.state).shape == (2, 3, V)


def _parents_of(history, prev):
    """Parent index of each beam of ``history`` [B, W, t] in ``prev`` [B, Wp, t-1]
    (the previous level's distinct beams) and its new token."""
    B, W, t = history.shape
    parents = torch.empty(B, W, dtype=torch.int64)
    for b in range(B):
        index = {tuple(s): i for i, s in enumerate(prev[b].tolist())}
        for w in range(W):
            parents[b, w] = index[tuple(history[b, w, :-1].tolist())]
    return parents, history[:, :, -1]


def test_tiny_grbeam_wide_level(device, tiny):
    """A level wider than the LDS-sorting merge (20,000 beams per request, on
    the workspace-sorting one), decoded and selected from again: widths
    [64, 20000, 4].  Level 0 equals the oracle's selection on the GPU's
    prefill logits; levels 1 and 2 are judged gap-aware against fp64 keys of
    the GPU's own logits (thousands of cross-row near-ties at the 20,000th
    key are ordered by fp32 rounding)."""
    from conftest import assert_selection_gap_aware

    cfg, oracle, adapter = tiny
    g = torch.Generator().manual_seed(23)
    ids = torch.randint(0, cfg.vocab_size, (2, 48), generator=g)
    two = grbeam_search(adapter, ids.to(device), [64, 20000])
    three = grbeam_search(adapter, ids.to(device), [64, 20000, 4])
    torch.cuda.synchronize()
    assert two.tokens.shape == (2, 20000, 2) and bool(two.valid.all())
    assert three.tokens.shape == (2, 4, 3) and bool(three.valid.all())
    h1 = two.tokens.cpu()
    for b in range(2):
        assert len({tuple(x) for x in h1[b].tolist()}) == 20000, "beams must be distinct"
    pre = adapter.prefill(ids.to(device))
    s0, p0, t0 = grbeam_ref.level_select(pre.logits.cpu()[:, None], torch.zeros(2, 1), 64)
    h0 = t0[..., None]
    logits1 = adapter.decode(h0.to(device), pre.state).cpu()
    keys1 = logits1.double().log_softmax(-1) + s0.double()[..., None]
    p1, t1 = _parents_of(h1, h0)   # every level-1 beam extends a level-0 beam
    assert_selection_gap_aware(two.scores.cpu(), p1, t1, keys1, 20000, delta=2e-5,
                               name="level 1")
    logits2 = adapter.decode(h1.to(device), pre.state).cpu()
    keys2 = logits2.double().log_softmax(-1) + two.scores.cpu().double()[..., None]
    p2, t2 = _parents_of(three.tokens.cpu(), h1)
    assert_selection_gap_aware(three.scores.cpu(), p2, t2, keys2, 4, delta=2e-5, name="level 2")


def test_reference_bf16_run_replayed_through_hip(device):
    """The reference's own bf16 search on the tiny model
    (tests/golden/grbeam_tiny_bf16.npz: the transformers bf16 prefill and the
    reference's bf16 decode, batch 1, prefix 128, widths [8, 8, 8]) replayed
    through the HIP adapter with the fixture's inputs at every level: the
    prefill and both decode levels' logits and every prefix tensor within rel
    1e-2 of the reference's, or (for tensors that compound several layers'
    bf16 rounding) no more than 10% farther from the fp32 evaluation of the
    same weights than the reference's own bf16 result is; at each level whose
    rank-W / W+1 key gap in the
    reference's own keys exceeds twice the measured largest logit error, the
    selected (parent, token) set equals the reference's; and where every level
    qualifies, grbeam_search returns the reference's tokens."""
    from _fixtures import bf16_from_bits, load_npz
    from kadllm_amd.grbeam import select_level

    f = load_npz("grbeam_tiny_bf16.npz")

    def t(name):
        a = f[name]
        return bf16_from_bits(a) if a.dtype == np.uint16 else torch.from_numpy(a)

    cfg = tiny_hybrid_config()
    sd = random_state_dict(cfg, seed=0, dtype=torch.bfloat16)   # the fixture's weights
    adapter = Qwen35GRBeamAdapter(*native_model(cfg, {k: v.to(device) for k, v in sd.items()}))
    ids = t("input_ids")
    widths = [int(w) for w in f["widths"]]
    pre = adapter.prefill(ids.to(device))
    torch.cuda.synchronize()
    truth = Qwen35Oracle(cfg, {k: v.float() for k, v in sd.items()})
    _, t_state = truth.prefill(ids)
    for i, (a, b) in enumerate(pre.state.layers):
        for j, (name, got) in enumerate((("a", a), ("b", b))):
            ref = t(f"prefix{i}_{name}")
            assert got.shape == ref.shape, (i, name, got.shape, ref.shape)
            r = rel_l2(got, ref)
            e_gpu, e_ref = rel_l2(got, t_state.layers[i][j]), rel_l2(ref, t_state.layers[i][j])
            print(f"prefix {i} {name}: rel L2 to the reference {r:.2e}; to fp32 truth: "
                  f"GPU {e_gpu:.2e}, reference {e_ref:.2e}", flush=True)
            assert r <= 1e-2 or e_gpu <= 1.1 * e_ref, f"prefix {i} {name}: rel L2 {r:.2e}"
    hist = [torch.empty(1, 1, 0, dtype=torch.int64), t("decode1_history"),
            t("decode2_history"), t("tokens")]
    ref_logits = [t("prefill_logits")[:, None], t("decode1_logits"), t("decode2_logits")]
    gpu_logits = [pre.logits[:, None]] + [adapter.decode(hist[s].to(device), pre.state)
                                          for s in (1, 2)]
    torch.cuda.synchronize()
    s_ref = torch.zeros(1, 1, dtype=torch.float64)
    s_gpu = torch.zeros(1, 1, device=device)
    all_levels = True
    exact = [truth.prefill(ids)[0][:, None]] + [truth.decode(hist[s], t_state) for s in (1, 2)]
    for step, W in enumerate(widths):
        g, r = gpu_logits[step], ref_logits[step]
        e = rel_l2(g, r)
        e_gpu, e_ref = rel_l2(g, exact[step]), rel_l2(r, exact[step])
        assert e <= 1e-2 or e_gpu <= 1.1 * e_ref, f"level {step}: logits rel L2 {e:.2e}"
        err = (g.float().cpu() - r.float()).abs().max().item()
        keys = (r.double().log_softmax(-1) + s_ref[..., None]).reshape(1, -1)
        top = torch.topk(keys, W + 1).values[0]
        gap = (top[W - 1] - top[W]).item()
        parents, tokens = _parents_of(hist[step + 1], hist[step])
        scores, p, tk, _ = select_level(g, s_gpu, W)
        torch.cuda.synchronize()
        decided = gap > 2 * err
        print(f"level {step}: logits rel L2 {e:.2e} (to fp32 truth: GPU {e_gpu:.2e}, reference "
              f"{e_ref:.2e}), max abs err {err:.3e}, rank-W/W+1 gap "
              f"{gap:.3e} -> {'compared' if decided else 'inside tolerance'}", flush=True)
        if decided:
            got = set(zip(p.cpu()[0].tolist(), tk.cpu()[0].tolist()))
            want = set(zip(parents[0].tolist(), tokens[0].tolist()))
            assert got == want, f"level {step}: selection differs from the reference's"
        all_levels &= decided
        # follow the reference's path: its beams (in its order) and scores
        flat = parents * r.shape[-1] + tokens
        s_ref = keys.gather(1, flat)
        order = [list(zip(p.cpu()[0].tolist(), tk.cpu()[0].tolist())).index(pt)
                 if decided else 0 for pt in zip(parents[0].tolist(), tokens[0].tolist())]
        s_gpu = scores[:, order] if decided else s_ref.float().to(device)
    if all_levels:
        result = grbeam_search(adapter, ids.to(device), widths)
        torch.cuda.synchronize()
        got = dict(zip(map(tuple, result.tokens.cpu()[0].tolist()), result.scores.cpu()[0].tolist()))
        want = dict(zip(map(tuple, t("tokens")[0].tolist()), t("scores")[0].tolist()))
        assert got.keys() == want.keys(), "search returns other beams than the reference's"
        for seq, sc in want.items():
            assert abs(got[seq] - sc) <= 3 * 2 * err + 1e-4, (seq, got[seq], sc)


@pytest.mark.parametrize("last", ["full_attention", "linear_attention"])
@pytest.mark.parametrize("B,L,W", [(1, 7, 10), (2, 128, 16), (3, 65, 5)])
def test_layers_in_one_call_equal_the_steps(device, last, B, L, W):
    """kad_qwen_prefill and kad_qwen_decode_step (one call per pass) against the
    runner's own steps, which a call hook brings back: logits, prefix and cache
    bit for bit, with the fused projection conv (L = 128) and without, kept and
    last levels, and a deep copy of the adapter."""
    import copy
    from dataclasses import replace

    from kadllm_amd import _lib
    cfg = replace(tiny_hybrid_config(), linear_key_head_dim=128, linear_value_head_dim=128,
                  layer_types=("linear_attention", "full_attention", "linear_attention", last))
    sd = random_state_dict(cfg, seed=4, dtype=torch.bfloat16, device=device)
    adapter = Qwen35GRBeamAdapter(*native_model(cfg, sd))
    g = torch.Generator().manual_seed(B * L)

    def ints(high, *shape):
        return torch.randint(0, high, shape, generator=g).to(device)

    ids, first = ints(cfg.vocab_size, B, L), ints(cfg.vocab_size, B, W, 1)
    parents, token = ints(W, B, W), ints(cfg.vocab_size, B, W, 1)
    second = torch.cat((first.gather(1, parents[..., None]), token), 2)

    def passes(ad):
        pre = ad.prefill(ids)
        l1, c1 = ad.decode_incremental(first, None, pre.state, None)
        l2, c2 = ad.decode_incremental(second, parents, pre.state, c1)
        l3, _ = ad.decode_incremental(second, parents, pre.state, c1, keep_cache=False)
        out = [pre.logits, l1, l2, l3, *(t for lyr in pre.state.layers for t in lyr)]
        for c in (c1, c2):
            for e in c.layers:
                # the projection rows' pad columns are never written
                out += list(e) if isinstance(e, tuple) else [e[:, :ad._runner.conv_dim
                                                               + ad._runner.vd]]
        return out

    names = []

    def hook(name, args, launch):
        names.append(name)
        launch()

    _lib.set_call_hook(hook)
    try:
        steps = passes(adapter)
    finally:
        _lib.set_call_hook(None)
    assert "kad_qwen_prefill" not in names and "kad_gemm_bf16" in names
    for ad in (adapter, copy.deepcopy(adapter)):
        for a, b in zip(passes(ad), steps):
            assert torch.equal(a, b)
    assert adapter._runner._native is not None


@pytest.mark.parametrize("HV", [2, 6, 4])
@pytest.mark.parametrize("W", [10, 16])
def test_last_level_of_any_value_head_count(device, HV, W):
    """A last level (no cache kept) whose gate rows, 4 HV bytes, are no whole
    16-byte pieces: the logits of the level that keeps its cache and of the whole
    suffix, as one call and step by step."""
    from dataclasses import replace

    from kadllm_amd import _lib
    B, L = 2, 9
    cfg = replace(tiny_hybrid_config(), linear_num_key_heads=2, linear_num_value_heads=HV,
                  linear_key_head_dim=128, linear_value_head_dim=128)
    adapter = Qwen35GRBeamAdapter(*native_model(cfg, random_state_dict(
        cfg, seed=5, dtype=torch.bfloat16, device=device)))
    g = torch.Generator().manual_seed(HV * W)

    def ints(high, *shape):
        return torch.randint(0, high, shape, generator=g).to(device)

    ids, first = ints(cfg.vocab_size, B, L), ints(cfg.vocab_size, B, W, 1)
    parents, token = ints(W, B, W), ints(cfg.vocab_size, B, W, 1)
    second = torch.cat((first.gather(1, parents[..., None]), token), 2)
    for hook in (None, lambda name, args, launch: launch()):
        _lib.set_call_hook(hook)
        try:
            state = adapter.prefill(ids).state
            _, cache = adapter.decode_incremental(first, None, state, None)
            kept, _ = adapter.decode_incremental(second, parents, state, cache)
            last, _ = adapter.decode_incremental(second, parents, state, cache, keep_cache=False)
            whole = adapter.decode(second, state)
        finally:
            _lib.set_call_hook(None)
        assert torch.equal(last, kept) and torch.equal(last, whole)


@pytest.mark.parametrize("how", ["rebound", "storage", "strided"])
def test_layers_in_one_call_follow_replaced_weights(device, how):
    """Weights of a layer replaced after a pass -- the attribute rebound, the
    tensor's storage exchanged, a tensor with strides of its own -- are those the
    next passes run with, as the single steps do."""
    from kadllm_amd import _lib
    cfg = tiny_hybrid_config()
    adapter = Qwen35GRBeamAdapter(*native_model(cfg, random_state_dict(
        cfg, seed=6, dtype=torch.bfloat16, device=device)))
    g = torch.Generator().manual_seed(6)
    ids = torch.randint(0, cfg.vocab_size, (2, 20), generator=g).to(device)
    tok = torch.randint(0, cfg.vocab_size, (2, 6, 1), generator=g).to(device)

    def logits():
        pre = adapter.prefill(ids)
        return pre.logits, adapter.decode_incremental(tok, None, pre.state, None)[0]

    before = logits()
    held = []                     # the old memory stays allocated throughout
    for lyr in (adapter._runner.layers[1], adapter._runner.layers[3]):
        for name in ("w_down", "post_norm"):
            old = getattr(lyr, name)
            new = old.flip(0).contiguous() * 0.5
            held.append(old if how != "storage" else old.data)
            if how == "storage":
                old.data = new
            elif how == "strided" and old.ndim == 2:
                wide = torch.zeros(old.shape[0], old.shape[1] + 64, dtype=old.dtype, device=device)
                setattr(lyr, name, wide[:, :old.shape[1]].copy_(new))
            else:
                setattr(lyr, name, new)
    got = logits()
    _lib.set_call_hook(lambda name, args, launch: launch())
    try:
        steps = logits()
    finally:
        _lib.set_call_hook(None)
    for b, a, e in zip(before, got, steps):
        assert torch.equal(a, e) and not torch.equal(a, b)
