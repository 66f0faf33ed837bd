"""Host-side mirror of the reference's layer call surface (transformer_models.py of the reference):
same class names, constructor arguments, state-dict keys, forward signatures and assertion behaviour,
with the arithmetic done by the HIP kernels of libterapipe_hip.so.

Differences that are deliberate: no ``mpu`` / ``torch.distributed`` process group is needed (tensor-
parallel size is 1, mpu/mappings.py:26-28 of the reference makes every collective an identity there);
the head dimension is one of 16, 32, 64, 80, 96, 128 (every entry of MODEL_CONFIGS); the K/V caches are written by the QKV GEMM's epilogue rather than by
a separate _AssignCache op, with the same in-place, alias-returning semantics and the same gradient
contract (reference transformer_models.py:177-193).
"""
import warnings
import weakref

import numpy as np
import torch
import torch.nn as nn
from torch.autograd import forward_ad
from torch.nn.modules import module as _modules

from . import _layer_core as core
from . import ops
from ._autograd import engine_adds_to_grad, fresh_leaves, note_leaves
from ._lib import TP_EPI_ACCUMULATE, TP_EPI_BIAS, TP_EPI_STORE, TP_GEMM_NN, TP_GEMM_NT, TP_GEMM_TN

# reference transformer_models.py:16 -- kept for callers that import it; the kernels mask by index.
NEG_INF = -65504

# name -> (n_layers, hidden_size, sequence_length, num_attention_heads); reference transformer_models.py:17-59
MODEL_CONFIGS = {
    "test": (24, 256, 128, 4),
    "test-l512": (512, 256, 128, 4),
    "test-s1024": (48, 2048, 1024, 32),
    "test-s2048": (48, 2048, 2048, 32),
    "test-h3072": (48, 3072, 2048, 48),
    "gpt2-1hm": (12, 768, 1024, 12),
    "gpt2-3hm": (24, 1024, 1024, 16),
    "gpt2-7hm": (36, 1280, 1024, 20),
    "gpt2-1b": (48, 1600, 1024, 25),
    "megatron-1b": (40, 1536, 1024, 16),
    "megatron-2b": (54, 1920, 1024, 20),
    "megatron-4b": (64, 2304, 1024, 24),
    "megatron-8b": (72, 3072, 1024, 32),
    "gpt3-1hm": (12, 768, 2048, 12),
    "gpt3-3hm": (24, 1024, 2048, 16),
    "gpt3-7hm": (24, 1536, 2048, 16),
    "gpt3-1b": (24, 2048, 2048, 16),
    "gpt3-2b": (32, 2560, 2048, 32),
    "gpt3-6b": (32, 4096, 2048, 32),
    "gpt3-13b": (40, 5120, 2048, 40),
    "gpt3-44b": (96, 6144, 2048, 48),
    "gpt3-175b": (96, 12288, 2048, 96),
    "gpt3-13b-4096": (40, 5120, 4096, 40),
    "gpt3-13b-6144": (40, 5120, 6144, 40),
    "gpt3-13b-8192": (40, 5120, 8192, 40),
    "gpt3-175b-megatron": (48, 6144, 2048, 384),
    "gpt2-1hm-single-device": (10, 768, 2048, 12),
    "gpt2-3hm-single-device": (8, 1024, 2048, 16),
    "gpt2-7hm-single-device": (6, 1280, 2048, 20),
    "gpt2-1b-single-device": (4, 1600, 2048, 25),
    "gpt3-1b-single-device": (5, 2048, 2048, 16),
    "gpt3-2b-single-device": (3, 2560, 2048, 32),
    "gpt3-6b-single-device": (2, 4096, 2048, 32),
    "gpt3-13b-single-device": (1, 5120, 2048, 40),
    "gpt3-175b-single-node": (2, 12288, 2048, 96),
}

# reference transformer_models.py:61-69
BATCH_CONFIGS = {"gpt3-1b": 72, "gpt3-13b": 32, "gpt3-44b": 16, "gpt3-175b": 2,
                 "gpt3-13b-4096": 8, "gpt3-13b-6144": 4, "gpt3-13b-8192": 2}


class TransformerConfig:
    """Shape bookkeeping of reference transformer_models.py:71-174 (single device: no placement)."""

    def __init__(self, batch_size=1, seq_len=1024, n_layers=12, embedding_dim=768, ffn_embedding_dim=None,
                 num_attention_heads=None, model_name=None):
        self.batch_size = batch_size
        if model_name is None:
            self.seq_len, self.n_layers, self.embedding_dim = seq_len, n_layers, embedding_dim
            self.ffn_embedding_dim = ffn_embedding_dim if ffn_embedding_dim else embedding_dim * 4
            self.num_attention_heads = num_attention_heads if num_attention_heads else embedding_dim // 64
        else:
            self.n_layers, self.embedding_dim, self.seq_len, self.num_attention_heads = MODEL_CONFIGS[model_name]
            self.ffn_embedding_dim = self.embedding_dim * 4

    @classmethod
    def from_predefined_model(cls, model_name, batch_size=1):
        return cls(batch_size=batch_size, model_name=model_name)

    @property
    def attention_heads_dim(self):
        return self.embedding_dim // self.num_attention_heads


# ------------------------------------------------------------------------------------------------
# linear layers (mpu/layers.py:193-353 of the reference at tensor-parallel size 1)
# ------------------------------------------------------------------------------------------------
class _LinearFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, bias):
        lead = x.shape[:-1]
        x2d = x.reshape(-1, x.shape[-1]).contiguous()
        M, K = x2d.shape
        N = weight.shape[0]
        y = torch.empty(M, N, dtype=x.dtype, device=x.device)
        if bias is not None:
            ops.gemm(TP_GEMM_NT, x2d, weight, M, N, K, C=y, epilogue=TP_EPI_BIAS, bias=bias)
        else:
            ops.gemm(TP_GEMM_NT, x2d, weight, M, N, K, C=y, epilogue=TP_EPI_STORE)
        ctx.save_for_backward(x2d, weight)
        ctx.has_bias = bias is not None
        ctx.lead = lead
        return y.view(*lead, N)

    @staticmethod
    def backward(ctx, dy):
        x2d, weight = ctx.saved_tensors
        M, K = x2d.shape
        N = weight.shape[0]
        dy2d = dy.reshape(M, N).contiguous()
        dx = torch.empty_like(x2d)
        ops.gemm(TP_GEMM_NN, dy2d, weight, M, K, N, C=dx)
        dw = torch.empty_like(weight)
        ops.gemm(TP_GEMM_TN, dy2d, x2d, N, K, M, C=dw)
        db = None
        if ctx.has_bias:
            acc = torch.zeros(N, dtype=torch.float32, device=dy.device)
            ops.colsum_acc(dy2d, acc)
            db = torch.empty(N, dtype=weight.dtype, device=dy.device)
            ops.accum_cast(db, acc, False)
        return dx.view(*ctx.lead, K), dw, db


class _ParallelLinearBase(nn.Module):
    def __init__(self, input_size, output_size, bias=True, init_method=nn.init.xavier_normal_, device="cuda"):
        super().__init__()
        self.input_size, self.output_size = input_size, output_size
        self.weight = nn.Parameter(torch.empty(output_size, input_size, device=device))   # [out, in]
        init_method(self.weight)
        if bias:
            self.bias = nn.Parameter(torch.zeros(output_size, device=device))              # always zero-init
        else:
            self.register_parameter("bias", None)

    def forward(self, input_):
        return _LinearFunction.apply(input_, self.weight, self.bias)


class ColumnParallelLinear(_ParallelLinearBase):
    """mpu.ColumnParallelLinear (reference mpu/layers.py:193-262) at tensor-parallel size 1:
    Y = X W^T + b, W stored [out, in], bias zero-initialised."""

    def __init__(self, input_size, output_size, bias=True, gather_output=True,
                 init_method=nn.init.xavier_normal_, device="cuda"):
        super().__init__(input_size, output_size, bias, init_method, device)
        self.gather_output = gather_output


class RowParallelLinear(_ParallelLinearBase):
    """mpu.RowParallelLinear (reference mpu/layers.py:265-353) at tensor-parallel size 1."""

    def __init__(self, input_size, output_size, bias=True, input_is_parallel=False,
                 init_method=nn.init.xavier_normal_, device="cuda"):
        super().__init__(input_size, output_size, bias, init_method, device)
        self.input_is_parallel = input_is_parallel


# ------------------------------------------------------------------------------------------------
# attention module and layer
# ------------------------------------------------------------------------------------------------
def _check_cache(full_cache, B, H, Dh, S, dtype):
    k, v = full_cache
    for c in (k, v):
        assert c.dim() == 3 and c.shape[0] == B * H and c.shape[2] == Dh, \
            "cache must be [batch*heads, seq_len, head_dim]"
        assert c.shape[1] >= S, "cache_len + slice length exceeds the cache"
        assert c.dtype == dtype and c.is_contiguous()
    return k, v


def _temp_cache(B, H, T, Dh, like):
    return (torch.empty(B * H, T, Dh, dtype=like.dtype, device=like.device),
            torch.empty(B * H, T, Dh, dtype=like.dtype, device=like.device))


def _grads_can_go_in_place(w):
    """Every parameter of the layer is a leaf with a dense .grad of its own dtype to add to, where the kernels can write it."""
    try:
        for p in w.values():
            g = p.grad if p.is_leaf else None
            if g is None or g.dtype is not p.dtype or g.shape != p.shape or not g.is_contiguous():
                return False
    except RuntimeError:        # (a sparse one is neither contiguous nor not)
        return False
    return not any(w[n].grad.data_ptr() % 16 for n in core.BIG_PARAMS)


class _GradOptions:
    """How a layer's backward hands its parameter gradients to autograd (TransformerLayer's two switches) and,
    for deferred weight gradients, the sequences under way (keyed by their K cache): the rows their forward has filled
    and the gradients of those whose backward runs."""
    __slots__ = ("in_place", "defer", "pending", "inputs")

    def __init__(self):
        self.in_place, self.defer, self.pending = False, False, {}
        self.inputs = weakref.WeakValueDictionary()     # the slices' graphs own them

    def __reduce__(self):
        # the switches are set anew by every forward, and a sequence under way belongs to the graphs of its slices: a copied
        # or unpickled layer starts with neither
        return _GradOptions, ()


class _SequenceInputs:
    """Deferred weight gradients: the inputs of the four linears of one sequence in one layer, position-indexed; the
    forward of a slice writes its rows (the next slice starts at `rows`)."""
    __slots__ = ("rows", "xn", "o", "hn", "a", "__weakref__")

    def __init__(self, rows, E, F, dtype, device):
        new = lambda n: torch.empty(rows, n, dtype=dtype, device=device)
        self.rows = 0
        self.xn, self.o, self.hn, self.a = new(E), new(E), new(E), new(F)


class _PendingGrads:
    """Deferred weight gradients of one sequence in one layer: the output gradients of the four linears for every
    position whose slice has run its backward (rows [low, rows); the reverse-slice order fills them from the end), and
    the fp32 sums of the vector-parameter gradients so far."""
    __slots__ = ("rows", "low", "inputs", "dqkv", "dh", "dz1", "dout", "acc")

    def __init__(self, rows, inputs, E, F, dtype, device):
        new = lambda n: torch.empty(rows, n, dtype=dtype, device=device)
        self.rows = self.low = rows
        self.inputs = inputs
        self.dqkv, self.dh, self.dz1, self.dout = new(3 * E), new(E), new(F), new(E)
        self.acc = torch.empty(core.small_acc_numel(E, F), dtype=torch.float32, device=device)


class _SliceKept:
    """The forward's kept activations as tensors, for whoever inspects a graph (the kernels work on addresses)."""
    __slots__ = ("geo", "arena", "seq", "cache_len")

    def __init__(self, geo, arena, seq, cache_len):
        self.geo, self.arena, self.seq, self.cache_len = geo, arena, seq, cache_len

    @property
    def a(self):
        g = self.geo
        if self.seq is not None:
            return self.seq.a[self.cache_len * g.B:self.cache_len * g.B + g.M]
        at = g.fwd.off["a"]
        return self.arena[at:at + g.M * g.F * g.es].view(g.dtype).view(g.M, g.F)


class _LayerFunction(torch.autograd.Function):
    """One whole layer over one slice.  Inputs: x, k_cache, v_cache (or None, None), then the 12
    parameters in core.PARAM_NAMES order.  Outputs: out, and the two caches when given.

    Forward and backward are one library call each (tp_layers_fwd, tp_layer_bwd).  The backward of a slice: the data
    gradients, the eight vector-parameter gradients as one launch, the four weight gradients as one grouped one.
    Where every parameter already has a .grad that the engine is going to add to on this node's stream
    (_autograd.engine_adds_to_grad), or with opts.in_place, the kernels add the gradients to it (the GEMM's accumulate
    epilogue, one rounding) and autograd gets None, instead of twelve tensors that autograd adds one elementwise kernel
    each.  opts.defer -- keep the slice's dY / X
    rows and take the weight gradients once per sequence, over all its rows, in the backward of the slice at position 0
    (the last one the reverse-slice order reaches); the slices before it hand autograd None for the parameters."""

    @staticmethod
    def forward(ctx, heads, cache_len, activation, opts, x, k_cache, v_cache, *params):
        T, B, E = x.shape
        ops._require_cuda(x, k_cache, v_cache)
        dt, dev = x.dtype, x.device
        F = params[8].shape[0]
        ctx.has_cache = k_cache is not None
        if not ctx.has_cache:
            k_cache, v_cache = _temp_cache(B, heads, T, E // heads, x)
        x = x.contiguous()
        geo = core.LayerGeometry.of(T, B, E, F, heads, dt, activation)
        out = torch.empty(T, B, E, dtype=dt, device=dev)
        seq, over = None, None
        if opts.defer and ctx.has_cache:
            # the slice's rows of the sequence's buffers; a slice that does not continue a sequence starts one
            r0, r1 = cache_len * B, (cache_len + T) * B
            key = k_cache.data_ptr()
            seq = opts.inputs.get(key)
            if seq is None or cache_len == 0 or seq.rows != r0 or seq.xn.shape[0] < r1:
                seq = None
                if cache_len == 0:
                    seq = opts.inputs[key] = _SequenceInputs(k_cache.shape[1] * B, E, F, dt, dev)
            if seq is not None:
                seq.rows = r1
                over = {n: getattr(seq, n)[r0:].data_ptr() for n in core.LINEAR_INPUTS}
        arena = torch.empty((geo.fwd_rest if over else geo.fwd).total, dtype=torch.uint8, device=dev)
        image = bytearray(core._FWD_PACK.size + core._BWD_PACK.size)
        geo.pack_fwd(image, 0, cache_len, k_cache.shape[1], params, x.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
                     arena.data_ptr(), out.data_ptr(), over)
        core.layers_fwd(image, 1, dev)
        ctx.geo, ctx.cache_len, ctx.opts = geo, cache_len, opts
        ctx.image = image               # the descriptor, for the backward to go on from (repack_operands)
        ctx.kept = (x, k_cache, v_cache, arena, seq)
        ctx.st = _SliceKept(geo, arena, seq, cache_len)
        ctx.w = params
        ctx.set_materialize_grads(False)
        if ctx.has_cache:
            # the caches were written through their raw pointers (as `cache.data[index] = value` does,
            # reference transformer_models.py:183); returning the inputs makes autograd hand back aliases
            return out, k_cache, v_cache
        return out

    @staticmethod
    def backward(ctx, dout, dk_out=None, dv_out=None):
        geo, opts, cache_len = ctx.geo, ctx.opts, ctx.cache_len
        x, k_cache, v_cache, arena, seq = ctx.kept
        w = dict(zip(core.PARAM_NAMES, ctx.w))
        T, B, E, F, M, dt, dev = geo.T, geo.B, geo.E, geo.F, geo.M, geo.dtype, x.device
        if dout is None:
            dout = torch.zeros(T, B, E, dtype=dt, device=dev)
        dout = dout.contiguous()
        gk, gv, gk_in, gv_in = _cache_grads(k_cache, dk_out, dv_out) if ctx.has_cache else (None,) * 4
        buf = torch.empty(geo.bwd.total, dtype=torch.uint8, device=dev)
        dx = torch.empty(T, B, E, dtype=dt, device=dev)
        base, off = buf.data_ptr(), geo.bwd.off
        p = {n: base + off[n] for n in off}
        fo, fbase = geo.fwd.off, arena.data_ptr()
        rows, dy = M, dout.data_ptr()
        pend, done, fresh = None, True, True
        if seq is not None:         # (deferred when its forward ran, whatever the switch says by now)
            # rows [r0, r1) of the sequence's position-indexed gradient buffers
            r0, r1 = cache_len * B, (cache_len + T) * B
            key = k_cache.data_ptr()
            pend = opts.pending.get(key)
            if pend is None or pend.low != r1 or pend.inputs is not seq:
                # the last slice of a sequence opens it; an entry that does not end where this slice begins belongs
                # to a sequence whose backward was abandoned or skipped a slice
                if pend is not None and pend.low < pend.rows:
                    warnings.warn("defer_weight_grads: the backward of a sequence stopped at row %d and never reached "
                                  "its first slice; its weight gradients are dropped" % pend.low)
                pend = opts.pending[key] = _PendingGrads(r1, seq, E, F, dt, dev)
            else:
                fresh = False
            p["dz1"], p["dh"], p["dqkv"] = (t[r0:].data_ptr() for t in (pend.dz1, pend.dh, pend.dqkv))
            p["small"] = pend.acc.data_ptr()
            if r1 - r0 < pend.rows:
                pend.dout[r0:r1].copy_(dout.view(M, E))
            else:
                pend.dout = dout                # the whole sequence in one slice
            pend.low = r0
            done = r0 == 0
            if done:
                del opts.pending[key]
                if opts.inputs.get(key) is seq:
                    del opts.inputs[key]
                rows = pend.rows
        in_place = done and _grads_can_go_in_place(w) and \
            (opts.in_place or engine_adds_to_grad(ctx, ctx.w, 3 if ctx.has_cache else 1))
        wg_out, small_out, wg = (0,) * 4, (0,) * 8, (0,) * 8
        grads = {}
        if done:
            if in_place:
                grads = {n: t.grad for n, t in w.items()}
            else:
                flat = torch.empty(geo.n_small, dtype=dt, device=dev)
                grads = core.small_acc_views(flat, E, F)
                for n in core.BIG_PARAMS:
                    grads[n] = torch.empty_like(w[n])
            wg_out = tuple(grads[n].data_ptr() for n in core.BIG_PARAMS)
            small_out = tuple(grads[n].data_ptr() for n in core.SMALL_PARAMS)
            if pend is not None:
                s = pend.inputs
                wg = (pend.dqkv.data_ptr(), s.xn.data_ptr(), pend.dh.data_ptr(), s.o.data_ptr(), pend.dz1.data_ptr(),
                      s.hn.data_ptr(), pend.dout.data_ptr(), s.a.data_ptr())
            else:
                xn, o, hn, a = (fbase + fo[n] for n in core.LINEAR_INPUTS)
                wg = (p["dqkv"], xn, p["dh"], o, p["dz1"], hn, dy, a)
        core.repack_operands(ctx.image, ctx.w, x, k_cache, v_cache)     # (a parameter's storage may have been replaced)
        core._BWD_PACK.pack_into(ctx.image, core._FWD_PACK.size, dy, p["dz1"], p["dhn"], p["dh"], p["d_o"], p["dqkv"],
                                 p["dxn"], dx.data_ptr(), p["delta"], p["small"],
                                 0 if gk is None else gk.data_ptr(), 0 if gv is None else gv.data_ptr(),
                                 geo.dt, 0, 0, 0, rows if done else 0, *wg, *wg_out,
                                 int(in_place), int(fresh), *small_out, int(in_place), int(ctx.has_cache),
                                 0 if gk_in is None else gk_in.data_ptr(), 0 if gv_in is None else gv_in.data_ptr())
        core.layer_bwd_native(ctx.image, dev)
        ctx.kept = ctx.image = ctx.w = ctx.st = None
        if not done or in_place:
            return (None, None, None, None, dx, gk, gv) + (None,) * len(core.PARAM_NAMES)
        return (None, None, None, None, dx, gk, gv) + tuple(grads[n] for n in core.PARAM_NAMES)


def _cache_grads(cache, dk_out, dv_out):
    """Gradients for the two cache inputs, not yet written, and those of the cache outputs as the kernel can read them (None
    where neither has one, zeros for one alone without).  The kernel leaves the latter as they are (grad_cache_output.clone(), reference
    transformer_models.py:188): it copies the rows that it does not add to."""
    gk, gv = (torch.empty_like(cache, memory_format=torch.contiguous_format) for _ in range(2))
    if dk_out is None and dv_out is None:
        return gk, gv, None, None
    if dk_out is None:
        dk_out = torch.zeros_like(dv_out)
    if dv_out is None:
        dv_out = torch.zeros_like(dk_out)
    # (the kernel's rows are contiguous and read 16 bytes at a time)
    return (gk, gv) + tuple(g if g.is_contiguous() and g.data_ptr() % 16 == 0 else
                            g.clone(memory_format=torch.contiguous_format) for g in (dk_out, dv_out))


class _AttentionFunction(torch.autograd.Function):
    """MultiheadLMAttentionWithCache alone: in_proj, cached attention, out_proj (+ bias)."""

    @staticmethod
    def forward(ctx, heads, cache_len, x, k_cache, v_cache, w_in, b_in, w_out, b_out):
        T, B, E = x.shape
        Dh = E // heads
        ctx.has_cache = k_cache is not None
        if not ctx.has_cache:
            k_cache, v_cache = _temp_cache(B, heads, T, Dh, x)
        w = {"attn.in_proj.weight": w_in, "attn.in_proj.bias": b_in}
        x2d = x.contiguous().view(T * B, E)
        q, o, lse = core.attention_fwd(w, x2d, T, B, heads, k_cache, v_cache, cache_len)
        y = torch.empty(T * B, E, dtype=x.dtype, device=x.device)
        ops.gemm(TP_GEMM_NT, o.view(T * B, E), w_out, T * B, E, E, C=y, epilogue=TP_EPI_BIAS, bias=b_out)
        ctx.saved = (x2d, q, o, lse, k_cache, v_cache, w_in, w_out)
        ctx.geom = (heads, cache_len, T, B, E, Dh)
        ctx.set_materialize_grads(False)
        if ctx.has_cache:
            return y.view(T, B, E), k_cache, v_cache
        return y.view(T, B, E)

    @staticmethod
    def backward(ctx, dy, dk_out=None, dv_out=None):
        x2d, q, o, lse, k_cache, v_cache, w_in, w_out = ctx.saved
        heads, cache_len, T, B, E, Dh = ctx.geom
        M = T * B
        if dy is None:
            dy = torch.zeros(T, B, E, dtype=x2d.dtype, device=x2d.device)
        dy2d = dy.contiguous().view(M, E)
        gk, gv, gk_in, gv_in = _cache_grads(k_cache, dk_out, dv_out) if ctx.has_cache else (None,) * 4
        acc = torch.zeros(4 * E, dtype=torch.float32, device=dy.device)
        acc_in, acc_out = acc[:3 * E], acc[3 * E:]
        d_o = torch.empty(M, E, dtype=dy.dtype, device=dy.device)
        ops.gemm(TP_GEMM_NN, dy2d, w_out, M, E, E, C=d_o)
        dw_out = torch.empty_like(w_out)
        ops.gemm(TP_GEMM_TN, dy2d, o.view(M, E), E, E, M, C=dw_out)
        ops.colsum_acc(dy2d, acc_out)
        dqkv = torch.empty(M, 3 * E, dtype=dy.dtype, device=dy.device)
        ops.attn_prefix_bwd(q, k_cache, v_cache, o, lse, d_o, dqkv, gk, gv, B, heads, Dh, T, cache_len,
                            float(Dh) ** -0.5, False, False, False, colsum_dqkv_acc=acc_in, whole_caches=ctx.has_cache,
                            dk_in=gk_in, dv_in=gv_in)
        dx = torch.empty(M, E, dtype=dy.dtype, device=dy.device)
        ops.gemm(TP_GEMM_NN, dqkv, w_in, M, E, 3 * E, C=dx)
        dw_in = torch.empty_like(w_in)
        ops.gemm(TP_GEMM_TN, dqkv, x2d, 3 * E, E, M, C=dw_in)
        db_in = torch.empty(3 * E, dtype=w_in.dtype, device=dy.device)
        db_out = torch.empty(E, dtype=w_in.dtype, device=dy.device)
        ops.accum_cast(db_in, acc_in, False)
        ops.accum_cast(db_out, acc_out, False)
        ctx.saved = None
        return None, None, dx.view(T, B, E), gk, gv, dw_in, db_in, dw_out, db_out


class MultiheadLMAttentionWithCache(nn.Module):
    """Reference transformer_models.py:196-261.  forward(x, full_cache=None, cache_len=0) returns
    (attn_out [T, B, E], (cache_k, cache_v) | None); the caches are updated in place on rows
    [cache_len, cache_len + T)."""

    def __init__(self, embed_dim, num_heads, bias=True, device="cpu"):
        super().__init__()
        self.embed_dim = embed_dim
        self.in_proj = ColumnParallelLinear(embed_dim, 3 * embed_dim, bias=bias, gather_output=False, device=device)
        self.out_proj = RowParallelLinear(embed_dim, embed_dim, bias=bias, input_is_parallel=True, device=device)
        if not bias:
            # the projection kernels fuse a bias: without one (reference transformer_models.py:197, :202-203)
            # they are given zeros, which are no parameters and appear in no state dict
            self.register_buffer("_no_in_bias", torch.zeros(3 * embed_dim, device=device), persistent=False)
            self.register_buffer("_no_out_bias", torch.zeros(embed_dim, device=device), persistent=False)
        self.num_heads = num_heads
        self.head_dim = embed_dim // num_heads
        assert self.head_dim * num_heads == self.embed_dim, "embed_dim must be divisible by num_heads"
        self.scaling = self.head_dim ** -0.5

    def forward(self, x, full_cache=None, cache_len=0, checkpoint_gradients=False):
        # checkpoint_gradients (reference checkpoint.py:24-43) needs no separate path: the attention
        # backward always recomputes the probabilities from q, k and the saved log-sum-exp.
        tgt_len, bsz, embed_dim = x.size()
        assert embed_dim == self.embed_dim
        k = v = None
        if full_cache is not None:
            k, v = _check_cache(full_cache, bsz, self.num_heads, self.head_dim, cache_len + tgt_len, x.dtype)
        else:
            assert cache_len == 0
        b_in = self.in_proj.bias if self.in_proj.bias is not None else self._no_in_bias
        b_out = self.out_proj.bias if self.out_proj.bias is not None else self._no_out_bias
        res = _AttentionFunction.apply(self.num_heads, cache_len, x, k, v, self.in_proj.weight, b_in,
                                       self.out_proj.weight, b_out)
        if full_cache is not None:
            return res[0], (res[1], res[2])
        return res, None

    def create_attn_cache(self, batch_size, seq_len, device="cuda", dtype=torch.float32):
        k = torch.zeros(batch_size * self.num_heads, seq_len, self.head_dim, device=device, dtype=dtype)
        v = torch.zeros(batch_size * self.num_heads, seq_len, self.head_dim, device=device, dtype=dtype)
        return k, v


class TransformerLayer(nn.Module):
    """Reference transformer_models.py:264-285: pre-LN block with a ReLU MLP.  (The reference's plain
    class omits `checkpoint_gradients` and cannot run; here it defaults to False.)"""

    # Two switches for loops that call .backward() / autograd.backward slice by slice, as the reference's does
    # (torch.autograd.grad would see None for the parameters, and post-accumulate-grad hooks may not fire):
    # accumulate_grads_in_place -- the backward of a slice adds its parameter gradients to existing .grad tensors
    # inside the gradient kernels instead of returning them to autograd (same sums, one rounding fewer), wherever it
    # runs: the caller keeps every forward of the layer, and its backward passes, on one stream;
    # defer_weight_grads -- with a cache, the weight gradients of a sequence are taken once, over all its rows, in
    # the backward of the slice at cache_len 0, which the reverse-slice order reaches last; .grad is complete when
    # that backward returns, and every slice of the sequence must run its backward, last slice first.
    accumulate_grads_in_place = False
    defer_weight_grads = False

    def __init__(self, embedding_dim, ffn_embedding_dim, num_attention_heads, device="cpu",
                 checkpoint_gradients=False, activation="relu"):
        super().__init__()
        self.checkpoint_gradients = checkpoint_gradients
        self.activation = activation
        self._grad_options = _GradOptions()
        self.attn_ln = nn.LayerNorm(embedding_dim).to(device)
        self.attn = MultiheadLMAttentionWithCache(embedding_dim, num_attention_heads, device=device)
        self.fc_ln = nn.LayerNorm(embedding_dim).to(device)
        self.fc1 = ColumnParallelLinear(embedding_dim, ffn_embedding_dim, gather_output=False, device=device)
        self.fc2 = RowParallelLinear(ffn_embedding_dim, embedding_dim, input_is_parallel=True, device=device)

    def param_list(self):
        """The 12 parameter tensors in core.PARAM_NAMES order."""
        try:
            # (straight from the modules' dictionaries: attribute look-ups through nn.Module cost as much as a launch)
            m = self._modules
            attn = m["attn"]._modules
            lin, out, fc1, fc2 = (t._parameters for t in (attn["in_proj"], attn["out_proj"], m["fc1"], m["fc2"]))
            ln1, ln2 = m["attn_ln"]._parameters, m["fc_ln"]._parameters
            return [ln1["weight"], ln1["bias"], lin["weight"], lin["bias"], out["weight"], out["bias"], ln2["weight"],
                    ln2["bias"], fc1["weight"], fc1["bias"], fc2["weight"], fc2["bias"]]
        except KeyError:        # a parametrized module computes its weight
            return [self.attn_ln.weight, self.attn_ln.bias, self.attn.in_proj.weight, self.attn.in_proj.bias,
                    self.attn.out_proj.weight, self.attn.out_proj.bias, self.fc_ln.weight, self.fc_ln.bias,
                    self.fc1.weight, self.fc1.bias, self.fc2.weight, self.fc2.bias]

    def param_dict(self):
        """The 12 parameter tensors keyed by their state-dict names."""
        return dict(zip(core.PARAM_NAMES, self.param_list()))

    def forward(self, x, full_cache=None, cache_len=0):
        tgt_len, bsz, embed_dim = x.shape
        attn = self._modules["attn"]
        assert embed_dim == attn.embed_dim
        k = v = None
        if full_cache is not None:
            k, v = _check_cache(full_cache, bsz, attn.num_heads, attn.head_dim, cache_len + tgt_len, x.dtype)
        else:
            assert cache_len == 0
        params = self.param_list()
        if not torch.is_grad_enabled() and not is_followed():
            # nothing to keep for a backward
            kv = (k, v) if k is not None else _temp_cache(bsz, attn.num_heads, tgt_len, attn.head_dim, x)
            out = core.stack_forward_only([(params, attn.num_heads, self.activation)], x, [kv], cache_len)
            return out, None if k is None else (k, v)
        opts = self._grad_options
        opts.in_place, opts.defer = bool(self.accumulate_grads_in_place), bool(self.defer_weight_grads)
        fresh = fresh_leaves(params)
        res = _LayerFunction.apply(attn.num_heads, cache_len, self.activation, opts, x, k, v, *params)
        if full_cache is not None:
            note_leaves(res[0].grad_fn, 3, fresh)
            return res[0], (res[1], res[2])
        note_leaves(res.grad_fn, 1, fresh)
        return res, None


def is_followed():
    """Whether somebody follows the computation node by node also without gradients: a trace records the layer as an autograd
    function, forward-mode differentiation has that function refuse."""
    return torch._C._get_tracing_state() is not None or forward_ad._current_level >= 0


def all_plain(layers):
    """Whether calling each of the modules is TransformerLayer.forward and nothing else: no subclass's or instance's own
    forward, no wrapper in a layer's place, no forward hooks (on a module or for all modules), not compiled.  A stack of such
    layers can run as one library call without anyone seeing the difference."""
    if _modules._global_forward_hooks or _modules._global_forward_pre_hooks:
        return False
    for layer in layers:
        kind, own = type(layer), layer.__dict__
        if (kind.forward is not TransformerLayer.forward or kind.__call__ is not nn.Module.__call__ or "forward" in own
                or own["_forward_hooks"] or own["_forward_pre_hooks"] or layer._compiled_call_impl is not None):
            return False
    return True


class ModelParallelMultiheadLMAttentionWithCache(MultiheadLMAttentionWithCache):
    """Reference transformer_models.py:288-311 at model-parallel size 1."""

    def __init__(self, embed_dim, num_heads, bias=True, device="cpu"):
        super().__init__(embed_dim, num_heads, bias=bias, device=device)
        self.model_parallel_size = 1
        self.num_total_heads = num_heads


class ModelParallelTransformerLayer(TransformerLayer):
    """Reference transformer_models.py:314-327 at model-parallel size 1 (the class the reference runs)."""

    def __init__(self, embedding_dim, ffn_embedding_dim, num_attention_heads, device="cpu",
                 checkpoint_gradients=False, activation="relu"):
        super().__init__(embedding_dim, ffn_embedding_dim, num_attention_heads, device=device,
                         checkpoint_gradients=checkpoint_gradients, activation=activation)
        self.model_parallel_size = 1


class SingleDeviceTransformer(nn.Module):
    """Reference transformer_models.py:330-342."""

    def __init__(self, transformer_layers):
        super().__init__()
        self.layers = nn.ModuleList(transformer_layers)

    def forward(self, x, attn_caches=None):
        if attn_caches is None:
            attn_caches = [None] * len(self.layers)
        new_attn_caches = []
        for layer, attn_cache in zip(self.layers, attn_caches):
            x, new_attn_cache = layer(x, attn_cache)
            new_attn_caches.append(new_attn_cache)
        return x, new_attn_caches


# ------------------------------------------------------------------------------------------------
# slicers (reference transformer_models.py:368-409)
# ------------------------------------------------------------------------------------------------
def uniform_slice_x(x, n_slices):
    seq_len = x.size(0)
    out, start = [], 0
    for i in range(n_slices):
        n = seq_len // n_slices + int(i < seq_len % n_slices)
        out.append(x[start:start + n])
        start += n
    assert start == seq_len
    return out


def grid_slice_batch_and_sequence(x, batch_slices, seq_slices, requires_grad=False, batch_dim=1, sequence_dim=0):
    """Object ndarray [n_batch_slices, n_seq_slices] of detached contiguous copies."""
    out = np.empty((len(batch_slices), len(seq_slices)), dtype="O")
    b0 = 0
    for i, bs in enumerate(batch_slices):
        s0 = 0
        for j, ss in enumerate(seq_slices):
            piece = x.narrow(sequence_dim, s0, ss).narrow(batch_dim, b0, bs)
            out[i, j] = piece.detach().contiguous().requires_grad_(requires_grad)
            s0 += ss
        assert s0 == x.size(sequence_dim)
        b0 += bs
    assert b0 == x.size(batch_dim)
    return out
