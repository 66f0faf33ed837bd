"""Functional core of one GPT layer over one sequence slice: the kernel sequence for forward and
backward, shared by the autograd wrappers in transformer_models.py and by the sliced runner in
terapipe.py.  Follows TransformerLayer.forward (transformer_models.py:273-285 of the reference) and
MultiheadLMAttentionWithCache.forward (:214-255); every arithmetic step is a call into
libterapipe_hip.so through terapipe_amd.ops.
"""
import ctypes
import struct

import torch

from . import _lib, ops
from ._lib import (TP_EPI_BIAS_GELU, TP_EPI_BIAS_RELU, TP_EPI_BIAS_RESIDUAL, TP_EPI_GELU_GRAD, TP_EPI_QKV_SCATTER,
                   TP_EPI_RELU_GRAD, TP_GEMM_NN, TP_GEMM_NT)

# order of the small (vector) parameters inside one layer's fp32 gradient accumulator
SMALL_PARAMS = ("attn_ln.weight", "attn_ln.bias", "attn.in_proj.bias", "attn.out_proj.bias",
                "fc_ln.weight", "fc_ln.bias", "fc1.bias", "fc2.bias")
BIG_PARAMS = ("attn.in_proj.weight", "attn.out_proj.weight", "fc1.weight", "fc2.weight")
PARAM_NAMES = ("attn_ln.weight", "attn_ln.bias", "attn.in_proj.weight", "attn.in_proj.bias",
               "attn.out_proj.weight", "attn.out_proj.bias", "fc_ln.weight", "fc_ln.bias",
               "fc1.weight", "fc1.bias", "fc2.weight", "fc2.bias")


def small_param_sizes(E, F):
    return {"attn_ln.weight": E, "attn_ln.bias": E, "attn.in_proj.bias": 3 * E, "attn.out_proj.bias": E,
            "fc_ln.weight": E, "fc_ln.bias": E, "fc1.bias": F, "fc2.bias": E}


def small_acc_views(buf, E, F):
    """Splits a flat fp32 buffer of small_acc_numel(E, F) elements into per-parameter views."""
    views, off = {}, 0
    for name in SMALL_PARAMS:
        n = small_param_sizes(E, F)[name]
        views[name] = buf[off:off + n]
        off += n
    return views


def small_acc_numel(E, F):
    return sum(small_param_sizes(E, F).values())


class SliceState:
    """What one layer keeps from the forward of one slice for its backward."""
    __slots__ = ("x", "mean1", "rstd1", "xn", "q", "o", "lse", "h", "mean2", "rstd2", "hn", "a", "z",
                 "k_cache", "v_cache", "cache_len", "T", "B", "q_bh_rows", "stat_bh_rows")


class Bufs:
    """Optional preallocated outputs for one layer-slice call (views into the runner's per-layer
    buffers).  Any attribute left at None is allocated by the call.  q_bh_rows / stat_bh_rows: q and
    lse / delta are views, starting at the slice's position, into position-indexed buffers with that many
    rows per (batch, head) -- 0 means compact [B*H, T, ...] tensors.  x_pending: the layer input is still the
    partial sums of the previous layer's k-split fc2 GEMM (ops.PendingReduce) and the first LayerNorm
    finishes it; defer_out: leave this layer's fc2 output in that state, returned in out_pending.
    sync: called (no arguments) at the one point of the layer where a slice depends on other slices: in forward
    after the in_proj GEMM has been launched and before the attention kernel (which reads the K/V rows the
    earlier slices' in_proj GEMMs write), in backward between the dQ kernel (which leaves this slice's delta)
    and the one-pass dK/dV kernel (which reads dO and delta of every later slice).  A runner that spreads
    slices over streams waits for / records its events there.  beside: other streams' launches run beside the call's."""
    __slots__ = ("xn", "mean1", "rstd1", "q", "o", "lse", "h", "mean2", "rstd2", "hn", "a", "z", "out",
                 "dz1", "dhn", "dh", "d_o", "dqkv", "dxn", "dx", "delta", "q_bh_rows", "stat_bh_rows",
                 "x_pending", "defer_out", "out_pending", "sync", "beside")

    def __init__(self, **kw):
        for n in self.__slots__:
            setattr(self, n, kw.get(n))
        self.q_bh_rows = self.q_bh_rows or 0
        self.stat_bh_rows = self.stat_bh_rows or 0


_NOBUF = Bufs()


def _buf(t, shape, dtype, device):
    return torch.empty(shape, dtype=dtype, device=device) if t is None else t


def attention_fwd(w, xn2d, T, B, heads, k_cache, v_cache, cache_len, buf=_NOBUF):
    """in_proj GEMM with the q/k/v split, q scaling and cache assignment fused into its epilogue, then
    the prefix-cached attention kernel.  Returns q [B*H, T, Dh], o [T, B, E], lse."""
    E = xn2d.shape[1]
    Dh = E // heads
    M = T * B
    q = _buf(buf.q, (B * heads, T, Dh), xn2d.dtype, xn2d.device)
    scale = float(Dh) ** -0.5
    ops.gemm(TP_GEMM_NT, xn2d, w["attn.in_proj.weight"], M, 3 * E, E, epilogue=TP_EPI_QKV_SCATTER,
             bias=w["attn.in_proj.bias"],
             qkv=dict(q=q, k_cache=k_cache, v_cache=v_cache, batch=B, heads=heads, head_dim=Dh,
                      cache_len=cache_len, cache_rows=k_cache.shape[1], q_scale=scale, q_bh_rows=buf.q_bh_rows),
             beside=buf.beside)
    if buf.sync is not None:
        buf.sync()
    o, lse = ops.attn_prefix_fwd(q, k_cache, v_cache, B, heads, Dh, T, cache_len, scale, out=buf.o, lse=buf.lse,
                                 q_bh_rows=buf.q_bh_rows, stat_bh_rows=buf.stat_bh_rows)
    return q, o, lse


def layer_fwd(w, x, heads, k_cache, v_cache, cache_len, activation="relu", need_state=True, buf=_NOBUF):
    """x [T, B, E] contiguous.  Writes rows [cache_len, cache_len+T) of the caches.  Returns (out, state)."""
    T, B, E = x.shape
    M = T * B
    F = w["fc1.weight"].shape[0]
    dt, dev = x.dtype, x.device
    x2d = x.view(M, E)
    xn, mean1, rstd1 = ops.layernorm_fwd(buf.x_pending if buf.x_pending is not None else x2d, w["attn_ln.weight"],
                                         w["attn_ln.bias"], out=buf.xn, mean=buf.mean1, rstd=buf.rstd1)
    q, o, lse = attention_fwd(w, xn, T, B, heads, k_cache, v_cache, cache_len, buf)
    o2d = o.view(M, E)
    h = _buf(buf.h, (M, E), dt, dev)
    # a k-split out_proj leaves its partial sums to the LayerNorm that follows directly (which then writes h)
    h_in = ops.gemm(TP_GEMM_NT, o2d, w["attn.out_proj.weight"], M, E, E, C=h, epilogue=TP_EPI_BIAS_RESIDUAL,
                    bias=w["attn.out_proj.bias"], residual=x2d, defer_reduce=True, beside=buf.beside)
    hn, mean2, rstd2 = ops.layernorm_fwd(h_in, w["fc_ln.weight"], w["fc_ln.bias"], out=buf.hn, mean=buf.mean2,
                                         rstd=buf.rstd2)
    a = _buf(buf.a, (M, F), dt, dev)
    z = None
    if activation == "relu":
        ops.gemm(TP_GEMM_NT, hn, w["fc1.weight"], M, F, E, C=a, epilogue=TP_EPI_BIAS_RELU, bias=w["fc1.bias"], beside=buf.beside)
    elif activation == "gelu":
        z = _buf(buf.z, (M, F), dt, dev)
        ops.gemm(TP_GEMM_NT, hn, w["fc1.weight"], M, F, E, C=a, epilogue=TP_EPI_BIAS_GELU, bias=w["fc1.bias"],
                 aux_out=z, beside=buf.beside)
    else:
        raise ValueError("activation must be 'relu' or 'gelu'")
    out = _buf(buf.out, (M, E), dt, dev)
    res = ops.gemm(TP_GEMM_NT, a, w["fc2.weight"], M, E, F, C=out, epilogue=TP_EPI_BIAS_RESIDUAL,
                   bias=w["fc2.bias"], residual=h, defer_reduce=bool(buf.defer_out), beside=buf.beside)
    if buf.defer_out:
        buf.out_pending = res if isinstance(res, ops.PendingReduce) else None
    st = None
    if need_state:
        st = SliceState()
        st.x, st.mean1, st.rstd1, st.xn = x2d, mean1, rstd1, xn
        st.q, st.o, st.lse = q, o2d, lse
        st.h, st.mean2, st.rstd2, st.hn = h, mean2, rstd2, hn
        st.a, st.z = a, z
        st.k_cache, st.v_cache, st.cache_len, st.T, st.B = k_cache, v_cache, cache_len, T, B
        st.q_bh_rows, st.stat_bh_rows = buf.q_bh_rows, buf.stat_bh_rows
    return out.view(T, B, E), st


def layer_bwd(w, st, dout, heads, gk, gv, accumulate_prefix, has_incoming, zero_slice_rows, activation="relu",
              buf=_NOBUF, suffix=None):
    """Backward of layer_fwd for one slice: the data gradients.

    dout [T, B, E]; gk / gv gradient caches (see tp_attn_desc).  The parameter gradients are the caller's: it
    keeps the intermediate gradients this call leaves in `buf` (dz1, dhn, dh, dqkv, dxn; dout is fc2's) and
    reduces them against the saved inputs -- per slice (the layer-level surface) or over all slices of a step at
    once (the runner): four TN products and eight column reductions (ops.gemm_grouped, ops.vec_param_grads).
    suffix: None, or dict(q_all, d_o_all, lse_all, delta_all, q_end) of position-indexed buffers that hold
    every slice processed so far (buf.d_o and buf.delta are then views of them at this slice): dK/dV of
    the slice's keys are computed in one pass over all later query positions and gk / gv are not used.
    With suffix["fused"] (needs o_all and own_end) dQ and that pass go out as one launch.
    Returns dx [T, B, E].
    """
    T, B = st.T, st.B
    M = T * B
    E = st.x.shape[1]
    F = st.a.shape[1]
    Dh = E // heads
    dt, dev = dout.dtype, dout.device
    dout2d = dout.reshape(M, E)
    # MLP
    dz1 = _buf(buf.dz1, (M, F), dt, dev)
    if activation == "relu":
        ops.gemm(TP_GEMM_NN, dout2d, w["fc2.weight"], M, F, E, C=dz1, epilogue=TP_EPI_RELU_GRAD, aux=st.a, beside=buf.beside)
    else:
        ops.gemm(TP_GEMM_NN, dout2d, w["fc2.weight"], M, F, E, C=dz1, epilogue=TP_EPI_GELU_GRAD, aux=st.z, beside=buf.beside)
    dhn = _buf(buf.dhn, (M, E), dt, dev)
    # a k-split data-gradient GEMM leaves its partial sums to the LayerNorm backward that follows directly
    dhn_in = ops.gemm(TP_GEMM_NN, dz1, w["fc1.weight"], M, E, F, C=dhn, defer_reduce=True, beside=buf.beside)
    dh = ops.layernorm_bwd(dhn_in, st.h, st.mean2, st.rstd2, w["fc_ln.weight"], dout2d, None, None, None, None,
                           out=buf.dh)
    # attention
    d_o = _buf(buf.d_o, (M, E), dt, dev)
    ops.gemm(TP_GEMM_NN, dh, w["attn.out_proj.weight"], M, E, E, C=d_o, beside=buf.beside)
    dqkv = _buf(buf.dqkv, (M, 3 * E), dt, dev)
    if suffix is None:
        ops.attn_prefix_bwd(st.q, st.k_cache, st.v_cache, st.o, st.lse, d_o, dqkv, gk, gv, B, heads, Dh, T,
                            st.cache_len, float(Dh) ** -0.5, accumulate_prefix, has_incoming, zero_slice_rows,
                            delta=buf.delta,
                            q_bh_rows=st.q_bh_rows, stat_bh_rows=st.stat_bh_rows)
    elif suffix.get("fused"):
        # dQ of the slice and dK / dV of its keys over all later positions as one launch.  The dK/dV half takes delta
        # of the positions up to own_end itself, so what it needs of the later slices is their dO (and, past own_end,
        # their delta): the slice waits for the next slice's event and records its own BEFORE the launch.  (An event
        # recorded there does not cover this launch's delta: the caller may only mix fused and two-launch slices
        # on ONE stream, see terapipe.fused_backward_slices.)
        if buf.sync is not None:
            buf.sync()
        ops.attn_bwd_fused(st.q, st.k_cache, st.v_cache, st.o, st.lse, d_o, dqkv, B, heads, Dh, T, st.cache_len,
                           float(Dh) ** -0.5, buf.delta, suffix["q_all"], suffix["d_o_all"], suffix["lse_all"],
                           suffix["delta_all"], suffix["o_all"], suffix["q_end"], suffix["own_end"],
                           q_bh_rows=st.q_bh_rows, stat_bh_rows=st.stat_bh_rows)
    else:
        ops.attn_prefix_bwd(st.q, st.k_cache, st.v_cache, st.o, st.lse, d_o, dqkv, None, None, B, heads, Dh, T,
                            st.cache_len, float(Dh) ** -0.5, False, False, False, delta=buf.delta,
                            q_bh_rows=st.q_bh_rows, stat_bh_rows=st.stat_bh_rows, dq_only=True)
        if buf.sync is not None:
            buf.sync()
        ops.attn_suffix_dkdv(st.k_cache, st.v_cache, suffix["q_all"], suffix["d_o_all"], suffix["lse_all"],
                             suffix["delta_all"], dqkv, B, heads, Dh, st.cache_len, T, suffix["q_end"])
    dxn = _buf(buf.dxn, (M, E), dt, dev)
    dxn_in = ops.gemm(TP_GEMM_NN, dqkv, w["attn.in_proj.weight"], M, E, 3 * E, C=dxn, defer_reduce=True, beside=buf.beside)
    dx = ops.layernorm_bwd(dxn_in, st.x, st.mean1, st.rstd1, w["attn_ln.weight"], dh, None, None, None, None,
                           out=buf.dx)
    return dx.view(T, B, E)


# ------------------------------------------------------------------------------------------------
# whole layers per library call (tp_layers_fwd, tp_layer_bwd): what the layer-level surface and the forward-only path use.
# A layer is nine to fifteen launches; issued one by one through ops.py each costs about 11 us of Python, which bounds
# short slices from the host.
# ------------------------------------------------------------------------------------------------
_FWD_PACK = struct.Struct("8iq28Q4q2i")        # tp_layer_desc: sizes, w[12], x, k_cache, v_cache, ..., ldw[4], no_backward
_FWD_READ, _FWD_LDW = struct.Struct("15Q"), struct.Struct("4q")
_FWD_READ_AT, _FWD_LDW_AT = 8 * 4 + 8, 8 * 4 + 8 + 28 * 8
_BWD_PACK = struct.Struct("12Q4iq8Q4Q2i8Q2i2Q")  # tp_layer_bwd_desc after its tp_layer_desc
_ACTIVATIONS = {"relu": 0, "gelu": 1}
LINEAR_INPUTS = ("xn", "o", "hn", "a")          # of in_proj, out_proj, fc1 and fc2


def operands(params, dtype):
    """(addresses, ldw) of a layer's 12 parameters in PARAM_NAMES order, as tp_layer_desc has them.  The library gets
    addresses only: what is not in GPU memory, not of the layer's type or not laid out as a kernel can read it is refused."""
    ldw = (0, 0, 0, 0)
    for p in params:
        if not (p.is_cuda and p.dtype is dtype and p.is_contiguous()):
            ldw = _row_pitches(params, dtype)
            break
    return [p.data_ptr() for p in params], ldw


def _row_pitches(params, dtype):
    """ldw where a weight may be a column range of a wider matrix."""
    ldw = [0, 0, 0, 0]
    for i, p in enumerate(params):
        ops._require_cuda(p)
        if p.dtype is not dtype:
            raise _lib.TeraPipeHipError("%s is %s, the layer's input %s" % (PARAM_NAMES[i], p.dtype, dtype))
        if not p.is_contiguous():
            if p.dim() != 2 or p.stride(1) != 1 or p.stride(0) < p.shape[1]:
                raise _lib.TeraPipeHipError("%s: strides %s; a vector, and each row of a weight, has to be contiguous"
                                            % (PARAM_NAMES[i], tuple(p.stride())))
            ldw[(2, 4, 8, 10).index(i)] = p.stride(0)
    return ldw


class _Arena:
    """Byte offsets (multiples of 256) of a set of buffers inside one allocation."""
    __slots__ = ("off", "total")

    def __init__(self, sizes):
        self.off, self.total = {}, 0
        for name, nbytes in sizes:
            self.off[name] = self.total
            self.total += (nbytes + 255) // 256 * 256


class LayerGeometry:
    """Sizes of one layer call and where its buffers lie.  Forward: what the backward reads again.  Backward: the
    intermediate gradients and the fp32 sums of the vector-parameter gradients."""
    __slots__ = ("T", "B", "E", "F", "H", "dtype", "es", "M", "activation", "fwd", "fwd_rest", "bwd", "n_small", "dt")
    _cache = {}

    def __init__(self, T, B, E, F, H, dtype, activation):
        self.T, self.B, self.E, self.F, self.H, self.dtype, self.activation = T, B, E, F, H, dtype, activation
        self.es, self.M, self.dt = dtype.itemsize, T * B, ops.tp_dtype(dtype)
        M, es = self.M, self.es
        rows = lambda width: M * width * es
        self.n_small = small_acc_numel(E, F)
        fwd = ([("xn", rows(E)), ("mean1", 4 * M), ("rstd1", 4 * M), ("q", rows(E)), ("o", rows(E)),
                ("lse", 4 * M * H), ("h", rows(E)), ("mean2", 4 * M), ("rstd2", 4 * M), ("hn", rows(E)),
                ("a", rows(F)), ("z", rows(F) if activation == "gelu" else 0)])
        # fwd_rest: without the inputs of the four linears, which a sequence with deferred weight gradients keeps
        self.fwd, self.fwd_rest = _Arena(fwd), _Arena([f for f in fwd if f[0] not in LINEAR_INPUTS])
        self.bwd = _Arena([("dz1", rows(F)), ("dhn", rows(E)), ("dh", rows(E)), ("d_o", rows(E)), ("dqkv", rows(3 * E)),
                           ("dxn", rows(E)), ("delta", 4 * M * H), ("small", 4 * self.n_small)])

    @classmethod
    def of(cls, T, B, E, F, H, dtype, activation):
        key = (T, B, E, F, H, dtype, activation)
        g = cls._cache.get(key)
        if g is None:
            if activation not in _ACTIVATIONS:
                raise ValueError("activation must be 'relu' or 'gelu'")
            if len(cls._cache) >= 512:
                cls._cache.clear()
            g = cls._cache[key] = cls(*key)
        return g

    def pack_fwd(self, image, at, cache_len, cache_rows, params, x, k, v, base, out, over=None, one_buffer=False,
                 no_backward=False):
        """Writes a tp_layer_desc at byte `at` of `image`.  params: the layer's 12; base: address of the forward arena; over: the
        addresses of LINEAR_INPUTS where they are not part of it (its layout is fwd_rest then).  one_buffer: for
        the rows of both LayerNorms.  no_backward: see tp_layer_desc."""
        w_ptrs, ldw = operands(params, self.dtype)
        o = (self.fwd_rest if over else self.fwd).off
        p = {n: base + o[n] for n in o}
        if over:
            p.update(over)
        if one_buffer:
            p["hn"] = p["xn"]
        _FWD_PACK.pack_into(image, at, self.dt, self.T, self.B, self.H, self.E, self.F, _ACTIVATIONS[self.activation],
                            cache_len, cache_rows, *w_ptrs, x, k, v, p["xn"], p["mean1"], p["rstd1"], p["q"], p["o"],
                            p["lse"], p["h"], p["mean2"], p["rstd2"], p["hn"], p["a"],
                            p["z"] if self.activation == "gelu" else 0, out, *ldw, int(no_backward), 0)


def repack_operands(image, params, x, k, v):
    """Writes into a packed tp_layer_desc where the parameters, the input and the caches are NOW."""
    w_ptrs, ldw = operands(params, x.dtype)
    _FWD_READ.pack_into(image, _FWD_READ_AT, *w_ptrs, x.data_ptr(), k.data_ptr(), v.data_ptr())
    _FWD_LDW.pack_into(image, _FWD_LDW_AT, *ldw)


def _address(image):
    return ctypes.addressof(ctypes.c_char.from_buffer(image))


def layers_fwd(images, n, device):
    """tp_layers_fwd on n packed descriptors, on the current stream."""
    lib = _lib.load()
    ptr = _address(images)
    stream = ops._stream()
    need = lib.tp_layers_fwd_workspace_bytes(ptr, n)
    ws = ops.Workspace.get(need, device, stream) if need else None
    _lib.check(lib.tp_layers_fwd(ptr, n, ops._p(ws), ws.numel() if ws is not None else 0, stream), "tp_layers_fwd")
    ops._record("layers_fwd", n, lambda s=None, ws=ws, keep=images: lib.tp_layers_fwd(
        ptr, n, ops._p(ws), ws.numel() if ws is not None else 0, ops._on(s)))


def layer_bwd_native(image, device):
    """tp_layer_bwd on a packed tp_layer_bwd_desc, on the current stream."""
    lib = _lib.load()
    ptr = _address(image)
    stream = ops._stream()
    need = lib.tp_layer_bwd_workspace_bytes(ptr)
    ws = ops.Workspace.get(need, device, stream) if need else None
    _lib.check(lib.tp_layer_bwd(ptr, ops._p(ws), ws.numel() if ws is not None else 0, stream), "tp_layer_bwd")
    ops._record("layer_bwd", 1, lambda s=None, ws=ws, keep=image: lib.tp_layer_bwd(
        ptr, ops._p(ws), ws.numel() if ws is not None else 0, ops._on(s)))


def stack_forward_only(layers, x, caches, cache_len):
    """The forward of a chain of layers without anything kept for a backward, as one library call: all layers share one
    set of intermediate buffers.  layers: [(12 parameters in PARAM_NAMES order, heads, activation)], each with its own
    FFN width, heads and activation; caches: [(k, v)] per layer.  Returns the output [T, B, E], the bits that the layers
    give under autograd: a forward without gradients may be recomputed with them (activation checkpointing), and half a
    rounding more or less turns ReLU units near zero on or off.  Only in inference mode, whose tensors autograd
    refuses, do products of a few rows take the forms that sum in another order."""
    T, B, E = x.shape
    ops._require_cuda(x, *(c for kv in caches for c in kv))
    x = x.contiguous()
    n = len(layers)
    known = {}
    geos = []
    for params, heads, activation in layers:
        kind = (params[8].shape[0], heads, activation)
        if kind not in known:
            known[kind] = LayerGeometry.of(T, B, E, kind[0], heads, x.dtype, activation)
        geos.append(known[kind])
    shared = max(g.fwd.total for g in known.values())
    step = (T * B * E * geos[0].es + 255) // 256 * 256
    # one allocation: the arena and, from two layers on, the outputs between the layers in turn
    arena = torch.empty(shared + (2 if n > 2 else n - 1) * step, dtype=torch.uint8, device=x.device)
    out = torch.empty_like(x)
    base = arena.data_ptr()
    image = bytearray(n * _FWD_PACK.size)
    src = x.data_ptr()
    for i, (params, _, _) in enumerate(layers):
        k, v = caches[i]
        dst = out.data_ptr() if i == n - 1 else base + shared + (i & 1) * step
        geos[i].pack_fwd(image, i * _FWD_PACK.size, cache_len, k.shape[1], params, src, k.data_ptr(), v.data_ptr(), base, dst,
                         one_buffer=n > 1, no_backward=torch.is_inference_mode_enabled())
        src = dst
    layers_fwd(image, n, x.device)
    return out
