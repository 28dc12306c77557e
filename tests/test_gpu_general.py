"""General-shape kernels (kad_gdn_recurrent, kad_attention_general, wide conv,
fp32/fp16 selection, beams above 1024) and the reference's toy model on them,
against the oracle and the reference's own outputs."""

import ctypes

import pytest
import torch

from kadllm_amd import _lib, grbeam_search, ops
from kadllm_amd.attention import prefix_attention_decode
from kadllm_amd.grbeam import select_level
from _fixtures import gdn_inputs
from conftest import assert_close_rel, assert_selection_gap_aware
from oracle import grbeam_ref, ops_ref
from test_oracle_reference_lm import reference_lm_case

pytestmark = pytest.mark.gpu


def _on(device, *ts):
    return [t.to(device) if t is not None else None for t in ts]


@pytest.mark.parametrize("dtype,B,W,T,H,HV,K,V", [
    (torch.float32, 2, 3, 7, 2, 2, 8, 8),
    (torch.float32, 1, 4, 9, 1, 2, 128, 128),   # past the factored replay's 8 tokens
    (torch.bfloat16, 2, 2, 5, 2, 4, 32, 48),
    (torch.float16, 2, 3, 3, 2, 2, 64, 64),
    (torch.float32, 1, 2, 2, 1, 1, 256, 70),
])
def test_gated_delta_general_matches_oracle(device, dtype, B, W, T, H, HV, K, V):
    q, k, v, g, beta, S = gdn_inputs(B, W, T, H, HV, K, V, dtype=dtype, seed=T + K)
    expected = ops_ref.gated_delta(q, k, v, g, beta, S, beam_width=W)
    S_dev = S.to(device)
    got = ops.gated_delta(*_on(device, q, k, v, g, beta), S_dev, beam_width=W)
    assert got.dtype == dtype
    if dtype == torch.float32:
        torch.testing.assert_close(got.cpu(), expected, atol=2e-5, rtol=1e-4)
    else:
        assert_close_rel(got, expected, rtol=1e-2, atol_frac=4e-3, name="gdn general")
    assert torch.equal(S_dev.cpu(), S)  # the prefix is read, never written


@pytest.mark.parametrize("dtype,K,V", [(torch.float32, 8, 8), (torch.float32, 64, 64),
                                       (torch.bfloat16, 16, 40)])
def test_gated_delta_final_state_general(device, dtype, K, V):
    B, W, T, H, HV = 2, 1, 9, 2, 2
    q, k, v, g, beta, S = gdn_inputs(B, W, T, H, HV, K, V, dtype=dtype, seed=3)
    eo, ef = ops_ref.gated_delta(q, k, v, g, beta, S, beam_width=W, return_final_state=True)
    go, gf = ops.gated_delta(*_on(device, q, k, v, g, beta, S), beam_width=W,
                             return_final_state=True)
    torch.testing.assert_close(gf.cpu(), ef, atol=2e-5, rtol=1e-4)
    if dtype == torch.float32:
        torch.testing.assert_close(go.cpu(), eo, atol=2e-5, rtol=1e-4)
    else:
        assert_close_rel(go, eo, rtol=1e-2, atol_frac=4e-3, name="gdn final")


@pytest.mark.parametrize("T", [1, 16, 17, 33])
@pytest.mark.parametrize("K,V,offset", [(1, 1, 0), (16, 17, 0), (33, 16, 0), (64, 15, 1),
                                        (128, 33, 0), (128, 16, 1), (256, 18, 0), (200, 5, 0)])
def test_gated_delta_recurrence_tile_edges(device, T, K, V, offset):
    """Tokens around the kernel's 16-token tiles, columns around its 16-column
    groups, key dims at and between its 16-lane splits, and rows that are not
    16-byte aligned (``offset`` elements into their storage).  fp32 sums of at
    most 256 terms over 33 steps of a contracting state: 2e-5 absolute."""
    q, k, v, g, beta, S = gdn_inputs(2, 1, T, 1, 2, K, V, dtype=torch.float32, seed=T + K)
    eo, ef = ops_ref.gated_delta(q.double(), k.double(), v.double(), g.double(), beta.double(),
                                 S.double(), return_final_state=True, compute=torch.float64)

    def shifted(t):
        d = torch.empty(t.numel() + offset, dtype=t.dtype, device=device)[offset:].view(t.shape)
        return d.copy_(t)

    go, gf = ops.gated_delta(*map(shifted, (q, k, v)), *_on(device, g, beta, S),
                             return_final_state=True)
    torch.testing.assert_close(go.double().cpu(), eo, atol=2e-5, rtol=1e-4)
    torch.testing.assert_close(gf.double().cpu(), ef.double(), atol=2e-5, rtol=1e-4)


def test_gated_delta_of_more_sequences_than_a_grid_holds(device):
    """2^24 + 3 one-token sequences of one-dimensional heads: as many workgroups of
    256, more work-items than one launch takes.  fp32: 1e-5 relative."""
    N = (1 << 24) + 3
    gen = torch.Generator(device=device).manual_seed(1)
    q, k, v, S = (torch.randn(N, 1, 1, 1, generator=gen, device=device) for _ in range(4))
    g = -torch.rand(N, 1, 1, generator=gen, device=device)
    beta = torch.rand(N, 1, 1, generator=gen, device=device)
    out, final = ops.gated_delta(q, k, v, g, beta, S, return_final_state=True)
    q, k, v, S, g, beta = (t.flatten().double() for t in (q, k, v, S, g, beta))
    kn = k / (k * k + 1e-6).sqrt()
    S = S * g.exp()
    S = S + kn * beta * (v - S * kn)
    torch.testing.assert_close(final.flatten().double(), S, atol=1e-5, rtol=1e-5)
    torch.testing.assert_close(out.flatten().double(), S * q / (q * q + 1e-6).sqrt(), atol=1e-5,
                               rtol=1e-5)


def _attn_inputs(B, W, T, H, HK, L, D, dtype, seed, Tk=None):
    g = torch.Generator().manual_seed(seed)
    Tk = T if Tk is None else Tk
    q = torch.randn(B * W, T, H, D, generator=g).to(dtype)
    pk = torch.randn(B, L, HK, D, generator=g).to(dtype)
    pv = torch.randn(B, L, HK, D, generator=g).to(dtype)
    sk = torch.randn(B * W, Tk, HK, D, generator=g).to(dtype)
    sv = torch.randn(B * W, Tk, HK, D, generator=g).to(dtype)
    return q, pk, pv, sk, sv


@pytest.mark.parametrize("dtype,B,W,T,H,HK,L,D", [
    (torch.float32, 2, 1, 5, 2, 2, 0, 8),       # a whole prompt, no prefix
    (torch.float32, 2, 3, 3, 4, 2, 17, 48),
    (torch.bfloat16, 1, 4, 10, 8, 2, 40, 256),  # suffix longer than the MFMA kernel's 8
    (torch.float32, 1, 2, 3, 4, 2, 20, 256),    # fp32 at head dim 256
    (torch.float16, 2, 2, 2, 4, 4, 33, 64),
    (torch.bfloat16, 2, 2, 3, 2, 1, 9, 96),     # head dim outside 64/128/256
])
def test_prefix_attention_general_matches_oracle(device, dtype, B, W, T, H, HK, L, D):
    q, pk, pv, sk, sv = _attn_inputs(B, W, T, H, HK, L, D, dtype, seed=L + D)
    mask = None
    if L:
        mask = torch.rand(B, L, generator=torch.Generator().manual_seed(5)) > 0.3
        mask[-1] = False  # a request whose prefix is fully masked
    expected = ops_ref.prefix_attention(q, pk, pv, sk, sv, beam_width=W, prefix_mask=mask)
    got = ops.prefix_attention(*_on(device, q, pk, pv, sk, sv), beam_width=W,
                               prefix_mask=_on(device, mask)[0])
    if dtype == torch.float32:
        torch.testing.assert_close(got.cpu(), expected, atol=2e-5, rtol=1e-4)
    else:
        assert_close_rel(got, expected, rtol=1e-2, atol_frac=4e-3, name="attention general")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("W,T,Tk,H,HK,L,D", [
    (5, 1, 1, 2, 2, 1, 64),      # 16-row tiles that end inside a request, one key
    (17, 1, 3, 4, 4, 16, 64),    # more beams than a tile's rows; a whole step of keys
    (3, 2, 2, 8, 2, 17, 256),
    (6, 3, 8, 8, 2, 65, 128),    # the longest suffix taken token by token
    (2, 9, 9, 8, 2, 33, 256),    # the shortest taken 16 tokens at a time
    (2, 2, 40, 8, 2, 0, 60),     # no prefix, a head dim of no whole vectors
    (1, 50, 50, 3, 1, 0, 256),   # a prompt whose rows straddle tokens
])
def test_prefix_attention_general_tile_edges(device, dtype, W, T, Tk, H, HK, L, D):
    """Rows against their own: the kernel's 16-row, 16-key steps and both suffix
    orders against the oracle, masked; and the last row's bits alone."""
    q, pk, pv, sk, sv = _attn_inputs(2, W, Tk, H, HK, L, D, dtype, seed=W + Tk + L)
    mask = torch.rand(2, L, generator=torch.Generator().manual_seed(L)) > 0.4 if L else None
    expected = ops_ref.prefix_attention(*(t.double() for t in (q, pk, pv, sk, sv)), beam_width=W,
                                        prefix_mask=mask)[:, Tk - T:]
    dev = _on(device, q[:, Tk - T:].contiguous(), pk, pv, sk, sv)
    got = prefix_attention_decode(*dev, W, _on(device, mask)[0], D ** -0.5)
    if dtype == torch.float32:
        torch.testing.assert_close(got.double().cpu(), expected, atol=2e-5, rtol=1e-4)
    else:  # half an ulp of the output, and of the inputs' 2^-11 products
        assert_close_rel(got, expected, rtol=2e-3, atol_frac=1e-3, name="attention tiles")
    last = prefix_attention_decode(dev[0][:, -1:].contiguous(), *dev[1:], W,
                                   _on(device, mask)[0], D ** -0.5)
    assert torch.equal(last, got[:, -1:])


@pytest.mark.parametrize("Tk", [2, 20])
def test_prefix_attention_general_nonfinite_values_stay_with_their_rows(device, Tk):
    """Infinite or NaN V entries reach only the rows that see their key: not
    through a mask, not into another beam, not before their position."""
    B, W, H, HK, L, D = 1, 4, 4, 2, 40, 64
    q, pk, pv, sk, sv = _attn_inputs(B, W, Tk, H, HK, L, D, torch.float32, seed=Tk)
    mask = torch.arange(L)[None] < 30
    pv[:, 30:] = float("nan")
    clean = sv.clone()
    sv[1, -1] = float("inf")
    expected = ops_ref.prefix_attention(q, pk, pv.nan_to_num(0.0), sk, clean, beam_width=W,
                                        prefix_mask=mask)
    got = ops.prefix_attention(*_on(device, q, pk, pv, sk, sv), beam_width=W,
                               prefix_mask=mask.to(device)).cpu()
    assert not torch.isfinite(got[1, -1]).any()
    got[1, -1] = expected[1, -1]
    torch.testing.assert_close(got, expected, atol=2e-5, rtol=1e-4)


def test_prefix_attention_of_more_rows_than_a_grid_holds(device):
    """2^20 + 1 requests of 16 heads and one token: 2^24 + 16 workgroups of 256,
    more work-items than one launch takes.  A row that sees one key is its V."""
    B, H, D = (1 << 20) + 1, 16, 4
    gen = torch.Generator(device=device).manual_seed(1)
    q, sk, sv = (torch.randn(B, 1, H, D, generator=gen, device=device) for _ in range(3))
    none = torch.empty(B, 0, H, D, device=device)
    assert torch.equal(ops.prefix_attention(q, none, none, sk, sv), sv)


@pytest.mark.parametrize("Tk", [2, 20])
def test_prefix_attention_general_rows_beside_nonfinite_ones_keep_their_bits(device, Tk):
    """A row whose result is not finite is computed again; the rows that share its
    tile are not: the bits of the same call without it."""
    B, W, H, HK, L, D = 1, 4, 4, 2, 40, 64
    dev = _on(device, *_attn_inputs(B, W, Tk, H, HK, L, D, torch.float32, seed=Tk))
    clean = ops.prefix_attention(*dev, beam_width=W)
    dev[0][1, -1] = 0.0
    dev[0][1, -1, :, 0] = float("inf")      # beam 1's last query: its scores and no others
    got = ops.prefix_attention(*dev, beam_width=W)
    assert not torch.isfinite(got[1, -1]).any()
    got[1, -1] = clean[1, -1]
    assert torch.equal(got, clean)


def test_prefix_attention_general_query_offset_and_gate(device):
    """Queries that are the last Tq of Tk suffix tokens equal the last rows of
    the full Tk-token attention; a gate multiplies by its rounded sigmoid."""
    B, W, H, HK, L, D, Tk, Tq = 2, 3, 4, 2, 20, 128, 7, 2
    q, pk, pv, sk, sv = _attn_inputs(B, W, Tk, H, HK, L, D, torch.bfloat16, seed=9)
    full = ops_ref.prefix_attention(q, pk, pv, sk, sv, beam_width=W)
    gate = torch.randn(B * W, Tq, H * D, generator=torch.Generator().manual_seed(2)).to(
        torch.bfloat16)
    got = prefix_attention_decode(*_on(device, q[:, Tk - Tq:].contiguous(), pk, pv, sk, sv), W,
                                  None, D ** -0.5, gate=gate.to(device))
    expected = (full[:, Tk - Tq:].float().reshape(B * W, Tq, H * D)
                * torch.sigmoid(gate.float()).bfloat16().float()).bfloat16()
    assert_close_rel(got.reshape(B * W, Tq, H * D), expected, rtol=1e-2, atol_frac=4e-3,
                     name="attention offset+gate")


@pytest.mark.parametrize("dtype,width,bias", [(torch.float32, 6, True), (torch.float16, 5, False),
                                              (torch.bfloat16, 8, True), (torch.float32, 3, True)])
def test_causal_conv1d_any_width(device, dtype, width, bias):
    g = torch.Generator().manual_seed(width)
    B, W, C, T = 2, 3, 24, 4
    x = torch.randn(B * W, C, T, generator=g).to(dtype)
    st = torch.randn(B, C, width + 1, generator=g).to(dtype)
    w = (torch.rand(C, width, generator=g) - 0.5).to(dtype)
    b = torch.randn(C, generator=g).to(dtype) if bias else None
    expected = ops_ref.causal_conv1d(x.float(), st.float(), w.float(), beam_width=W,
                                     bias=None if b is None else b.float())
    got = ops.causal_conv1d(*_on(device, x, st, w), beam_width=W, bias=_on(device, b)[0])
    tol = {torch.float32: 1e-5, torch.float16: 2e-3, torch.bfloat16: 1.6e-2}[dtype]
    torch.testing.assert_close(got.float().cpu(), expected, atol=tol, rtol=tol)


def test_triton_conv_backend_requires_width4_silu_nobias(device):
    x = torch.randn(2, 8, 2, device=device, dtype=torch.bfloat16)
    st = torch.randn(2, 8, 3, device=device, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="Triton short-conv requires width=4, SiLU, and no bias"):
        ops.causal_conv1d(x, st, torch.randn(8, 3, device=device, dtype=torch.bfloat16),
                          backend="triton")
    with pytest.raises(ValueError, match="Triton short-conv"):
        ops.causal_conv1d(x, st, torch.randn(8, 4, device=device, dtype=torch.bfloat16),
                          activation=None, backend="triton")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("B,Wp,V,width,masked", [
    (2, 3, 4095, 40, False),     # rows that are candidates whole, at odd offsets
    (1, 2, 4097, 1500, True),
    (2, 3, 60001, 300, True),    # sampled, every row at another alignment
    (1, 520, 9001, 9, False),    # more rows than two per CU: 256 threads a row
    (1, 2, 300000, 256, False),
])
def test_select_rows_of_any_length(device, dtype, B, Wp, V, width, masked):
    """The row stage over its ways in: rows below and above the candidate
    buffer, misaligned rows, both workgroup sizes, masks.  Scores 1e-5 from the
    64-bit log-softmax (fp32 sums of up to 300,000 terms)."""
    g = torch.Generator().manual_seed(V + width)
    logits = (torch.randn(B, Wp, V, generator=g) * 2).to(dtype)
    scores = -torch.rand(B, Wp, generator=g) * 3
    mask = torch.rand(B, Wp, V, generator=g) > 0.5 if masked else None
    s, p, t, valid = select_level(logits.to(device), scores.to(device), width,
                                  None if mask is None else mask.to(device))
    keys = logits.double().log_softmax(-1) + scores.double()[..., None]
    if masked:
        keys = keys.masked_fill(~mask, -float("inf"))
    assert bool(valid.all())
    assert_selection_gap_aware(s, p, t, keys, width, 1e-5, name="rows")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("V,where", [(1001, "head"), (60001, "unsampled")])
def test_select_rows_whose_sample_holds_no_finite_logit(device, dtype, V, where):
    """Rows whose finite logits, near -120, are all in the columns before the
    row's first 16-byte boundary, or in lines the sample leaves out (with as many
    allowed -inf ones in it): the sum's reference is 0 there, against which every
    term underflows.  Scores 1e-5 from the 64-bit log-softmax."""
    g = torch.Generator().manual_seed(V)
    Wp, W = 4, 3
    logits = torch.full((1, Wp, V), -float("inf"))
    finite = torch.zeros(V, dtype=torch.bool)
    allowed = torch.zeros(V, dtype=torch.bool)
    if where == "head":
        finite[:3] = True
        allowed[:] = True
    else:
        finite[100:300] = True      # lines 2 .. 4 of every 7
        allowed = finite.clone()
        allowed[64 * 7 * torch.arange(1, 121) + 20] = True
    logits[0, :, finite] = -120 + torch.randn(Wp, int(finite.sum()), generator=g)
    logits = logits.to(dtype)
    scores = -torch.rand(1, Wp, generator=g)
    mask = allowed.expand(1, Wp, V)
    s, p, t, valid = select_level(logits.to(device), scores.to(device), W, mask.to(device))
    keys = (logits.double().log_softmax(-1) + scores.double()[..., None])
    keys = keys.masked_fill(~mask, -float("inf"))
    assert bool(valid.all())
    assert_selection_gap_aware(s, p, t, keys, W, 1e-5, name="rows")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("peak", [18.0, 30.0, 60.0])
def test_select_float_scores_under_a_peak_outside_the_sample(device, dtype, peak):
    """A confident model's rows: Gaussian logits and one far above them, in a line
    the sample leaves out.  The peak's key is -lse alone: its thread adds some 60
    words' sums to 1, half an ulp each in either direction (worst case 30 ulps,
    sqrt(60) / 2 expected, twice that allowed); the others' keys are three
    roundings more, half an ulp each."""
    Wp, V, W = 8, 248320, 24
    logits = torch.randn(1, Wp, V, generator=torch.Generator().manual_seed(int(peak)))
    logits[0, torch.arange(Wp), 70 + 3 * torch.arange(Wp)] = peak
    logits = logits.to(dtype)
    s, p, t, valid = select_level(logits.to(device), torch.zeros(1, Wp, device=device), W)
    keys = logits.double().log_softmax(-1)
    true = keys[0, p[0].cpu(), t[0].cpu()]
    err = (s[0].double().cpu() - true).abs()
    top = t[0].cpu() == 70 + 3 * p[0].cpu()
    assert int(top.sum()) == Wp and bool(valid.all())
    ulp = 2.0 ** (true.abs().clamp_min(1.0).log2().floor() - 23)
    assert bool((err[top] <= 8 * 2.0 ** -23).all()), err[top]
    assert bool((err[~top] <= 1.5 * ulp[~top] + 8 * 2.0 ** -23).all()), err[~top]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("allowed", [0, 1, 20, 700, 3000, 9000])
@pytest.mark.parametrize("spread", ["block", "random"])
def test_select_rows_of_few_allowed_columns(device, dtype, allowed, spread):
    """Constraint masks that leave a block of columns, or as many anywhere: fewer
    than the level's width, than the sample's rank, than the candidate buffer,
    and more.  Unfilled slots take the lowest masked candidates, in order."""
    Wp, V, W = 5, 60001, 40
    g = torch.Generator().manual_seed(allowed)
    logits = (torch.randn(1, Wp, V, generator=g) * 2).to(dtype)
    scores = -torch.rand(1, Wp, generator=g)
    mask = torch.zeros(1, Wp, V, dtype=torch.bool)
    for r in range(Wp):
        at = torch.randperm(V, generator=g)[:allowed] if spread == "random" else \
            torch.arange(20000 + 900 * r, 20000 + 900 * r + allowed)
        mask[0, r, at] = True
    s, p, t, valid = select_level(logits.to(device), scores.to(device), W, mask.to(device))
    keys = (logits.double().log_softmax(-1) + scores.double()[..., None])
    keys = keys.masked_fill(~mask, -float("inf"))
    n = min(W, Wp * allowed)
    assert int(valid.sum()) == n and bool(valid[0, :n].all())
    if n:
        assert_selection_gap_aware(s[:, :n], p[:, :n], t[:, :n], keys, n, 1e-5, name="few")
    free = (~mask[0]).reshape(-1).nonzero()[:W - n, 0]
    assert torch.equal((p * V + t)[0, n:].cpu(), free)


def test_select_float_rows_with_equal_keys_take_lower_columns(device):
    """fp32 logits that differ by less than their keys' precision tie, and the
    lower columns of all of them are taken, sampled or not."""
    V, W = 50000, 20
    logits = torch.full((1, 1, V), -3.0)         # one value: every key equal
    s, p, t, _ = select_level(logits.to(device), torch.zeros(1, 1, device=device), W)
    assert t[0].tolist() == list(range(W))
    logits[0, 0, 40000:40010] = 1e-6             # logits apart, keys (near -7.8) equal
    logits[0, 0, 40000:40010] += torch.arange(10) * 1e-9
    s, p, t, _ = select_level(logits.to(device), torch.zeros(1, 1, device=device), 4)
    assert t[0].tolist() == [40000, 40001, 40002, 40003]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_select_float_logits_matches_oracle(device, dtype):
    g = torch.Generator().manual_seed(11)
    B, Wp, V, width = 3, 5, 1000, 7
    logits = (torch.randn(B, Wp, V, generator=g) * 3).to(dtype)
    scores = torch.randn(B, Wp, generator=g)
    mask = torch.rand(B, Wp, V, generator=g) > 0.2
    for m in (None, mask):
        es, ep, et = grbeam_ref.level_select(logits, scores, width, m)
        s, p, t, valid = select_level(*_on(device, logits, scores), width,
                                      None if m is None else m.to(device))
        assert torch.equal(p.cpu(), ep) and torch.equal(t.cpu(), et)
        torch.testing.assert_close(s.cpu(), es, atol=1e-5, rtol=1e-6)
        assert bool(valid.all())


@pytest.mark.parametrize("B,Wp,V,width", [(2, 4, 2048, 3000), (1, 16, 4096, 16384)])
def test_select_beams_above_1024(device, B, Wp, V, width):
    """Widths past the 1024 the merge once held, up to its LDS limit.  Judged
    gap-aware against fp64 keys: thousands of picks sit within fp32 noise of
    picks from other rows, whose order rounding decides."""
    g = torch.Generator().manual_seed(width)
    logits = torch.randn(B, Wp, V, generator=g).bfloat16()
    scores = torch.randn(B, Wp, generator=g)
    s, p, t, valid = select_level(*_on(device, logits, scores), width)
    keys = logits.double().log_softmax(-1) + scores.double()[..., None]
    assert_selection_gap_aware(s, p, t, keys, width, delta=2e-5, name=f"W={width}")
    assert bool(valid.all())


@pytest.mark.parametrize("B,Wp,V,width", [(1, 3, 12000, 20000), (2, 40, 2048, 40000)])
def test_select_beams_above_lds_limit(device, B, Wp, V, width):
    """Widths past the LDS-sorting merge (16,384) take the workspace-sorting
    one; judged gap-aware against fp64 keys as the narrower widths are."""
    g = torch.Generator().manual_seed(width + Wp)
    logits = torch.randn(B, Wp, V, generator=g).bfloat16()
    scores = torch.randn(B, Wp, generator=g)
    s, p, t, valid = select_level(*_on(device, logits, scores), width)
    keys = logits.double().log_softmax(-1) + scores.double()[..., None]
    assert_selection_gap_aware(s, p, t, keys, width, delta=2e-5, name=f"W={width}")
    assert bool(valid.all())


def test_select_wide_exact_ties_and_mask(device):
    """One row per request with a handful of distinct logit values, so the
    20,000th pick falls inside a class of equal keys: ties go to the lower
    column, exactly as the oracle orders them; masked entries score -inf and
    rank last."""
    g = torch.Generator().manual_seed(5)
    B, Wp, V, width = 2, 1, 60000, 20000
    logits = (torch.randint(-4, 5, (B, Wp, V), generator=g).float() / 2).bfloat16()
    scores = torch.zeros(B, Wp)
    mask = torch.rand(B, Wp, V, generator=g) > 0.5
    for m in (None, mask):
        es, ep, et = grbeam_ref.level_select(logits, scores, width, m)
        s, p, t, valid = select_level(*_on(device, logits, scores), width,
                                      None if m is None else m.to(device))
        assert torch.equal(p.cpu(), ep) and torch.equal(t.cpu(), et)
        fin = torch.isfinite(es)
        assert torch.equal(valid.cpu(), fin)
        torch.testing.assert_close(s.cpu()[fin], es[fin], atol=1e-5, rtol=0)


@pytest.mark.parametrize("B,Wp,V,width", [(3, 5, 1000, 7), (2, 8, 4096, 3000),
                                          (2, 16, 2048, 16384)])
def test_wide_merge_equals_lds_merge(device, B, Wp, V, width):
    """The two request-level kernels on the same row candidates (logits with
    many exact ties) give the same picks, scores and order, bit for bit."""
    from kadllm_amd import _lib
    from kadllm_amd.grbeam import merge

    g = torch.Generator().manual_seed(width)
    logits = (torch.randint(-20, 21, (B, Wp, V), generator=g).float() / 4).bfloat16().to(device)
    parent = torch.randint(-3, 1, (B, Wp), generator=g).float().to(device)
    K = min(width, V)
    cand_key = torch.empty(B * Wp, K, dtype=torch.float32, device=device)
    cand_idx = torch.empty(B * Wp, K, dtype=torch.int32, device=device)
    stream = _lib.stream_of(logits)
    _lib.call("kad_beam_row_select", _lib.ptr(logits), 0, V, None, V, _lib.ptr(parent),
              B * Wp, Wp, V, K, _lib.ptr(cand_key), _lib.ptr(cand_idx), stream)
    outs = []
    for wide in (False, True):
        o = (torch.empty(B, width, device=device), torch.empty(B, width, dtype=torch.int64,
                                                                device=device),
             torch.empty(B, width, dtype=torch.int64, device=device),
             torch.empty(B, width, dtype=torch.bool, device=device))
        merge(cand_key, cand_idx, B, Wp * K, width, V, *o, stream, wide=wide)
        outs.append([x.cpu() for x in o])
    for a, b in zip(*outs):
        assert torch.equal(a, b)


def test_reference_hybrid_lm_readme_example(device):
    """README.md:254-266: ReferenceHybridLM(vocab_size=32), prompts [2, 5],
    widths [2, 3, 4] gives tokens [2, 4, 3]."""
    from kadllm import grbeam_search as search
    from kadllm.adapters import ReferenceHybridLM

    torch.manual_seed(0)
    model = ReferenceHybridLM(vocab_size=32).to(device).eval()
    prompts = torch.randint(0, 32, (2, 5), device=device)
    with torch.inference_mode():
        result = search(model, prompts, widths=[2, 3, 4])
    assert tuple(result.tokens.shape) == (2, 4, 3)
    assert bool(result.valid.all())


@pytest.mark.parametrize("ci", [0, 1])
def test_reference_hybrid_lm_matches_reference_outputs(device, ci):
    """The HIP toy model with the reference's weights reproduces the reference's
    search: tokens exactly, scores and every level's logits within fp32 noise."""
    from kadllm.adapters import ReferenceHybridLM

    c = reference_lm_case(ci)
    model = ReferenceHybridLM(vocab_size=c["vocab"], hidden_size=c["hidden"],
                              num_heads=c["heads"])
    model.load_state_dict(c["sd"])
    model = model.to(device).eval()
    seen = []
    decode = model.decode

    def recording(history, state):
        out = decode(history, state)
        seen.append((history.cpu(), out.cpu()))
        return out

    model.decode = recording
    result = grbeam_search(model, c["ids"].to(device), c["widths"])
    with torch.no_grad():
        pre = model.prefill(c["ids"].to(device))
    torch.testing.assert_close(pre.logits.cpu(), c["prefill_logits"], atol=1e-4, rtol=1e-4)
    assert len(seen) == len(c["calls"])
    for (h, got), (eh, expected) in zip(seen, c["calls"]):
        assert torch.equal(h, eh)
        torch.testing.assert_close(got, expected, atol=1e-4, rtol=1e-4)
    assert torch.equal(result.tokens.cpu(), c["tokens"])
    torch.testing.assert_close(result.scores.cpu(), c["scores"], atol=1e-4, rtol=1e-5)
    assert torch.equal(result.valid.cpu(), c["valid"])


@pytest.mark.parametrize("B,L,N,C,K", [(2, 128, 1024, 768, 256), (3, 256, 512, 256, 128),
                                       (1, 1024, 1024, 512, 64), (2, 256, 8192, 6144, 1024)])
def test_gemm_conv_prefill_equals_gemm_then_conv(device, B, L, N, C, K):
    """kad_gemm_bf16_conv against kad_gemm_bf16 followed by
    kad_causal_conv_prefill, bit for bit: the conv columns, the plain columns
    past them, and the conv state; sequences of one and of several 128-row
    blocks per tile, a wider output row stride (the last case is the GDN
    input projection of the 0.8B model)."""
    M = B * L
    g = torch.Generator().manual_seed(M + N + C + K)
    a = (torch.randn(M, K, generator=g) * 0.5).bfloat16().to(device)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16().to(device)
    cw = (torch.rand(C, 4, generator=g) - 0.5).bfloat16().to(device)
    ldc = N + 64
    stream = _lib.stream_of(a)
    plain = torch.empty(M, N, dtype=torch.bfloat16, device=device)
    _lib.call("kad_gemm_bf16", _lib.ptr(a), K, _lib.ptr(w), K, _lib.ptr(plain), N, None, 0, M, N, K,
              0, stream)
    conv = torch.empty(M, C, dtype=torch.bfloat16, device=device)
    st1 = torch.empty(B, C, 4, dtype=torch.bfloat16, device=device)
    _lib.call("kad_causal_conv_prefill", _lib.ptr(plain), N, _lib.ptr(cw), _lib.ptr(conv), C,
              _lib.ptr(st1), B, L, C, 1, stream)
    nb = ctypes.c_int64(0)
    _lib.call("kad_gemm_bf16_conv_workspace_bytes", M, C, ctypes.byref(nb))
    ws = torch.empty(nb.value, dtype=torch.uint8, device=device)
    out = torch.full((M, ldc), 9.0, dtype=torch.bfloat16, device=device)
    st2 = torch.empty(B, C, 4, dtype=torch.bfloat16, device=device)
    _lib.call("kad_gemm_bf16_conv", _lib.ptr(a), K, _lib.ptr(w), K, _lib.ptr(out), ldc, M, N, K, C,
              _lib.ptr(cw), L, _lib.ptr(st2), _lib.ptr(ws), ws.numel(), stream)
    torch.cuda.synchronize()
    assert torch.equal(out[:, :C], conv), "fused conv columns differ"
    assert torch.equal(out[:, C:N], plain[:, C:]), "plain columns differ"
    assert torch.equal(st2, st1), "conv state differs"
    assert (out[:, N:].float() == 9.0).all(), "wrote past N"


def test_gemm_conv_prefill_rejects_unsupported(device):
    """Shapes off the fused form are refused (the model then makes the two calls)."""
    a = torch.zeros(256, 64, dtype=torch.bfloat16, device=device)
    w = torch.zeros(512, 64, dtype=torch.bfloat16, device=device)
    cw = torch.zeros(256, 4, dtype=torch.bfloat16, device=device)
    out = torch.empty(256, 512, dtype=torch.bfloat16, device=device)
    ws = torch.empty(1 << 20, dtype=torch.uint8, device=device)
    # sequences of 64 rows; conv columns not a multiple of 256
    for L, C in ((64, 256), (128, 128)):
        with pytest.raises(_lib.KadLibraryError, match="unsupported"):
            _lib.call("kad_gemm_bf16_conv", _lib.ptr(a), 64, _lib.ptr(w), 64, _lib.ptr(out), 512,
                      256, 512, 64, C, _lib.ptr(cw), L, None, _lib.ptr(ws), ws.numel(),
                      _lib.stream_of(a))
