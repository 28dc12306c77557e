"""One foreign call per pass of a bf16 model's layers (kad_qwen_prefill,
kad_qwen_decode_step): the structs of include/kadllm_hip.h and the buffers they
name.  The kernels, their order and arguments are those of Qwen35Runner's own
loops, which run where a trace or a call hook wants every step, and for the
shapes outside ``step_fits``."""

import ctypes
import operator

import torch

from . import _lib

_P, _I, _L, _F = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_float


class _Layer(ctypes.Structure):
    _fields_ = [("linear", _I)] + [(n, _P) for n in (
        "input_norm", "post_norm", "w_gu", "w_down", "w_in", "w_ab", "conv_w", "A_log", "dt_bias",
        "norm_w", "w_out", "w_qkv", "q_norm", "k_norm", "w_o")]


class _Model(ctypes.Structure):
    _fields_ = [("layers", ctypes.POINTER(_Layer)), ("inv_freq", _P)] + [(n, _I) for n in (
        "n_layers", "hidden", "ffn", "conv_dim", "kd", "vd", "gdn_cols", "ab_rows", "k_heads",
        "v_heads", "k_dim", "v_dim", "q_heads", "kv_heads", "head_dim", "rot")] + [
        ("eps", _F), ("gdn_scale", _F), ("attn_scale", _F)]


class _PrefillArgs(ctypes.Structure):
    _fields_ = [(n, _I) for n in ("layers", "B", "L", "fuse_conv")] + [(n, _P) for n in (
        "state0", "state1", "x", "n", "h", "proj", "mixed", "q", "beta", "conv", "chunk_ws",
        "g")] + [("conv_bytes", _L), ("chunk_bytes", _L)]


class _Prefix(ctypes.Structure):
    _fields_ = [("p0", _P), ("p1", _P), ("s0", _L), ("s1", _L), ("s2", _L), ("history", _I),
                ("dtype", _I)]


class _StepArgs(ctypes.Structure):
    _fields_ = [(n, _I) for n in ("B", "W", "Wp", "T", "keep", "prefetch")] + [("pos", _L)] + [
        (n, _P) for n in ("parents", "prefix", "prev0", "prev1", "next0", "next1", "x", "n", "h",
                          "mixed", "q", "qkv", "rows_ws", "k_ws", "v_ws", "ab", "beta", "g")]


def _pointers(tensors):
    """A C array of device addresses (null for None)."""
    return (_P * len(tensors))(*[None if t is None else t.data_ptr() for t in tensors])


_COMMON = ("input_norm", "post_norm", "w_gu", "w_down")
_LINEAR = _COMMON + ("w_in", "w_ab", "conv_w", "A_log", "dt_bias", "norm_w", "w_out")
_ATTENTION = _COMMON + ("w_qkv", "q_norm", "k_norm", "w_o")
_get_linear, _get_attention = operator.attrgetter(*_LINEAR), operator.attrgetter(*_ATTENTION)


def _weights(runner):
    """Every tensor whose address kad_qwen_model holds."""
    out = [runner.inv_freq]
    for lyr in runner.layers:
        out += _get_linear(lyr) if hasattr(lyr, "w_in") else _get_attention(lyr)
    return out


class NativeLayers:
    """The packed weights of a Qwen35Runner as kad_qwen_model, and its passes."""

    def __init__(self, runner):
        cfg = runner.cfg
        layers = (_Layer * len(runner.layers))()
        self.linear = []
        for dst, src in zip(layers, runner.layers):
            dst.linear = int(hasattr(src, "w_in"))
            self.linear.append(bool(dst.linear))
            for name in _LINEAR if dst.linear else _ATTENTION:
                setattr(dst, name, getattr(src, name).data_ptr())
        # the tensors are held, so that no address outlives its memory
        self._layers, self._tensors = layers, _weights(runner)
        self._addresses = list(map(torch.Tensor.data_ptr, self._tensors))
        # the passes name no strides and no types
        self.plain = all(t.is_contiguous() and t.dtype == (
            torch.float32 if t is runner.inv_freq else torch.bfloat16) for t in self._tensors)
        self.ab_rows = 2 * cfg.linear_num_value_heads
        self.ffn = runner.layers[0].w_down.shape[1]
        # one width throughout (the padded packing of every layer's MLP)
        self.uniform = all(lyr.w_down.shape[1] == self.ffn for lyr in runner.layers)
        self.model = _Model(
            layers, runner.inv_freq.data_ptr(), len(runner.layers), cfg.hidden_size, self.ffn,
            runner.conv_dim, runner.kd, runner.vd, runner.gdn_cols, self.ab_rows,
            cfg.linear_num_key_heads, cfg.linear_num_value_heads, cfg.linear_key_head_dim,
            cfg.linear_value_head_dim, cfg.num_attention_heads, cfg.num_key_value_heads,
            cfg.head_dim, runner.rot, cfg.rms_norm_eps, cfg.linear_key_head_dim ** -0.5,
            cfg.head_dim ** -0.5)
        self.qkv_cols = runner.attn_cols
        self.att_cols = cfg.num_attention_heads * cfg.head_dim
        # the fused decode mixer's and the MFMA attention's shapes
        self.step_shapes = (
            self.uniform and cfg.linear_key_head_dim == 128 and cfg.linear_value_head_dim == 128
            and runner.gdn_cols % 8 == 0 and cfg.linear_num_value_heads % 2 == 0
            and cfg.head_dim in (64, 128, 256)
            and all(lyr.conv_w.is_contiguous() and lyr.conv_w.data_ptr() % 8 == 0
                    and lyr.norm_w.data_ptr() % 8 == 0
                    for lyr, lin in zip(runner.layers, self.linear) if lin))

    def describes(self, runner):
        """Whether the runner's weights are still the tensors, at the addresses,
        that the struct was built from (a layer's may be rebound or its storage
        replaced): 25 us for 24 layers."""
        now = _weights(runner)
        return (len(now) == len(self._tensors)
                and all(map(operator.is_, now, self._tensors))
                and list(map(torch.Tensor.data_ptr, now)) == self._addresses)

    def _call(self, name, args, x):
        _lib.call(name, ctypes.addressof(self.model), ctypes.addressof(args), _lib.stream_of(x))

    def prefill(self, runner, x, B, L, count):
        """The first ``count`` layers over x [B*L, hidden] in place; returns
        their prefix tensors."""
        cfg, dev, rows = runner.cfg, x.device, B * L
        C, HV = runner.conv_dim, cfg.linear_num_value_heads
        dk, dv = cfg.linear_key_head_dim, cfg.linear_value_head_dim
        nkv, hd = cfg.num_key_value_heads, cfg.head_dim

        def empty(*shape, dtype=torch.bfloat16):
            return torch.empty(*shape, dtype=dtype, device=dev)

        state0, state1 = [], []
        for lin in self.linear[:count]:
            if lin:
                state0.append(empty(B, C, 4))
                state1.append(empty(B, HV, dk, dv, dtype=torch.float32))
            else:
                state0.append(empty(B, nkv, L, hd))
                state1.append(empty(B, nkv, L, hd))
        gdn = any(self.linear[:count])
        fuse = gdn and all(runner.conv_fuses(rows, L, lyr) for lyr, lin in
                           zip(runner.layers[:count], self.linear) if lin)
        if fuse:
            nb = _L(0)
            _lib.call("kad_gemm_bf16_conv_workspace_bytes", rows, C, ctypes.byref(nb))
            conv = torch.empty(nb.value, dtype=torch.uint8, device=dev)
        else:
            conv = empty(rows, C) if gdn else None
        ws = _lib.gdn_chunk_workspace(B, L, HV, dk, dev) if gdn else x
        n, h = empty(rows, cfg.hidden_size), empty(rows, self.ffn)
        proj = empty(rows, max(runner.gdn_cols, self.qkv_cols))
        mixed = empty(rows, max(runner.vd, self.att_cols))
        q, g = empty(rows, self.att_cols), empty(rows, HV, dtype=torch.float32)
        beta = empty(rows, HV)
        s0, s1 = _pointers(state0), _pointers(state1)
        ptr = torch.Tensor.data_ptr
        args = _PrefillArgs(
            count, B, L, int(fuse), ctypes.addressof(s0), ctypes.addressof(s1), ptr(x), ptr(n),
            ptr(h), ptr(proj), ptr(mixed), ptr(q), ptr(beta), _lib.ptr(conv), ptr(ws), ptr(g),
            conv.numel() if fuse else 0, ws.numel() if gdn else 0)
        self._call("kad_qwen_prefill", args, x)
        return [(a, b) if lin else (a.transpose(1, 2), b.transpose(1, 2))
                for a, b, lin in zip(state0, state1, self.linear)]

    def step_fits(self, T, prefix_layers):
        """Whether kad_qwen_decode_step takes this level: two tokens at most,
        attention prefixes it can read in place."""
        if not self.step_shapes or T > 2:
            return False
        for (a, b), lin in zip(prefix_layers, self.linear):
            if a.dtype != torch.bfloat16:
                return False
            if lin:
                if not b.is_contiguous():
                    return False
            elif (a.stride() != b.stride() or a.stride(3) != 1 or a.shape[1] < 1
                  or any(s % 8 for s in a.stride()[:3]) or b.dtype != torch.bfloat16
                  or a.data_ptr() % 16 or b.data_ptr() % 16):
                return False
        return True

    def decode_step(self, runner, x, B, W, T, Wp, parents, prefix_layers, prefix_length, cache,
                    keep, prefetch):
        """All layers over x [B*W, hidden] in place; returns the level's cache
        entries (empty without ``keep``)."""
        cfg, dev, BW = runner.cfg, x.device, B * W
        HV, nkv, hd = cfg.linear_num_value_heads, cfg.num_key_value_heads, cfg.head_dim
        cols = runner.gdn_cols

        def empty(*shape, dtype=torch.bfloat16):
            return torch.empty(*shape, dtype=dtype, device=dev)

        prefix = (_Prefix * len(self.linear))()
        for dst, (a, b), lin in zip(prefix, prefix_layers, self.linear):
            dst.p0, dst.p1 = a.data_ptr(), b.data_ptr()
            dst.s0, dst.s1, dst.s2 = a.stride()[:3]
            dst.history = a.shape[2] if lin else a.shape[1]
            dst.dtype = _lib.dtype_code(b.dtype)
        new = []
        if keep:
            new = [empty(BW * T, cols) if lin else (empty(BW, T, nkv, hd), empty(BW, T, nkv, hd))
                   for lin in self.linear]

        def split(entries):
            return (_pointers([e if lin else e[0] for e, lin in zip(entries, self.linear)]),
                    _pointers([None if lin else e[1] for e, lin in zip(entries, self.linear)]))

        arrays = [split(cache.layers) if T > 1 else (None, None),
                  split(new) if keep else (None, None)]
        at = [None if p is None else ctypes.addressof(p) for pair in arrays for p in pair]
        n, h = empty(BW, cfg.hidden_size), empty(BW, self.ffn)
        mixed, q = empty(BW, max(runner.vd, self.att_cols)), empty(BW, self.att_cols)
        # a last level reads the earlier token's rows in its parents' cache where
        # the gate inputs are whole 16-byte pieces, else gathers all T of a beam
        parent_rows = T == 1 or keep or self.ab_rows % 8 == 0
        qkv, rows_ws = empty(BW, self.qkv_cols), empty(BW * (1 if parent_rows else T), cols)
        k_ws, v_ws = (None, None) if keep else (empty(BW, T, nkv, hd), empty(BW, T, nkv, hd))
        ab, beta = empty(BW * T, self.ab_rows), empty(BW * T, HV)
        g = empty(BW * T, HV, dtype=torch.float32)
        ptr = _lib.ptr
        args = _StepArgs(B, W, Wp, T, int(keep), int(prefetch), prefix_length, ptr(parents),
                         ctypes.addressof(prefix), *at, ptr(x), ptr(n), ptr(h), ptr(mixed), ptr(q),
                         ptr(qkv), ptr(rows_ws), ptr(k_ws), ptr(v_ws), ptr(ab), ptr(beta), ptr(g))
        self._call("kad_qwen_decode_step", args, x)
        return new
