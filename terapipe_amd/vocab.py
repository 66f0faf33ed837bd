"""The two ends of the layer stack at tensor-parallel size 1: token embedding, LM head, vocabulary
cross-entropy.  Mirrors mpu.VocabParallelEmbedding (reference mpu/layers.py:85-141) and
mpu.vocab_parallel_cross_entropy (mpu/cross_entropy.py:25-110); every arithmetic step is a call into
libterapipe_hip.so through terapipe_amd.ops.
"""
import torch
import torch.nn as nn
from torch.nn import init

from . import ops
from ._autograd import lookup_to_hand_to, note_lookup, taken_on
from ._lib import TP_EPI_ACCUMULATE, TP_EPI_STORE, TP_GEMM_NN, TP_GEMM_NT, TP_GEMM_TN


class _EmbeddingFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, ids, weight):
        flat = ids.reshape(-1).contiguous()
        out = ops.embedding_fwd(flat, weight)
        ctx.save_for_backward(flat)
        ctx.wshape, ctx.wdtype = weight.shape, weight.dtype
        return out.view(*ids.shape, weight.shape[1])

    @staticmethod
    def backward(ctx, dout):
        """The rows that occur are added to the gradient that an LM head tied to this weight has handed over (no dense
        gradient of the lookup is made then, and none is added), otherwise to zeros."""
        (flat,) = ctx.saved_tensors
        dout = dout.reshape(flat.numel(), -1).contiguous()
        handed = taken_on(ctx)
        if ops.embedding_rows_fit(flat, dout):
            dw = torch.zeros(ctx.wshape, dtype=ctx.wdtype, device=dout.device) if handed is None else handed
            return None, ops.embedding_bwd_rows_(flat, dout, dw)
        acc = torch.empty(ctx.wshape, dtype=torch.float32, device=dout.device)
        ops.zero_(acc)
        ops.embedding_bwd(flat, dout, acc)
        if handed is None and ctx.wdtype == torch.float32:
            return None, acc
        dw = torch.empty(ctx.wshape, dtype=ctx.wdtype, device=dout.device) if handed is None else handed
        ops.accum_cast(dw, acc, handed is not None)
        return None, dw


class VocabParallelEmbedding(nn.Module):
    """mpu.VocabParallelEmbedding at tensor-parallel size 1 (the vocabulary range is the whole vocabulary,
    mpu/layers.py:108-113; the all-reduce of :139 is the identity)."""

    def __init__(self, num_embeddings, embedding_dim, init_method=init.xavier_normal_, device=None, dtype=None):
        super().__init__()
        self.num_embeddings, self.embedding_dim = num_embeddings, embedding_dim
        self.padding_idx, self.max_norm, self.norm_type = None, None, 2.0
        self.scale_grad_by_freq, self.sparse = False, False
        self.vocab_start_index, self.vocab_end_index = 0, num_embeddings
        self.num_embeddings_per_partition = num_embeddings
        self.weight = nn.Parameter(torch.empty(num_embeddings, embedding_dim, device=device, dtype=dtype))
        init_method(self.weight)

    def forward(self, input_):
        out = _EmbeddingFunction.apply(input_, self.weight)
        if out.grad_fn is not None:
            note_lookup(out.grad_fn, 1)
        return out


VOCAB_PAD = 64      # logits rows are whole 128-byte lines


def _pad_vocab(n):
    return (n + VOCAB_PAD - 1) // VOCAB_PAD * VOCAB_PAD


def _as_operand(weight):
    """The weight where a GEMM can read it: itself, or a copy where it is strided or not 16-byte aligned."""
    weight = weight.contiguous()
    return weight.clone() if weight.data_ptr() % 16 else weight


class _LMHeadFunction(torch.autograd.Function):
    """logits = h W^T, rows padded to a multiple of 64 columns (zeros; the loss ignores them)."""

    @staticmethod
    def forward(ctx, h2d, weight):
        V, E = weight.shape
        Vp = _pad_vocab(V)
        h2d = h2d.contiguous()
        logits = torch.empty(h2d.shape[0], Vp, dtype=h2d.dtype, device=h2d.device)
        ops.gemm(TP_GEMM_NT, h2d, _as_operand(weight), h2d.shape[0], V, E, C=logits, epilogue=TP_EPI_STORE,
                 ragged=True)
        if Vp != V:
            logits[:, V:].zero_()
        ctx.save_for_backward(h2d, weight)
        return logits

    @staticmethod
    def backward(ctx, dlogits):
        h2d, weight = ctx.saved_tensors
        M, E = h2d.shape
        V = weight.shape[0]
        dlogits = dlogits.contiguous()
        dh = torch.empty_like(h2d)
        ops.gemm(TP_GEMM_NN, dlogits, _as_operand(weight), M, E, V, C=dh, ragged=True)
        tied = lookup_to_hand_to(ctx, 1)        # an embedding of the same weight adds its rows to what it is handed
        if tied is not None and tied.handed is not None:
            ops.gemm(TP_GEMM_TN, dlogits, h2d, V, E, M, C=tied.handed, epilogue=TP_EPI_ACCUMULATE, ragged=True)
            return dh, None
        dw = torch.empty(weight.shape, dtype=weight.dtype, device=weight.device)
        ops.gemm(TP_GEMM_TN, dlogits, h2d, V, E, M, C=dw, ragged=True)
        if tied is not None:
            tied.handed = dw
            return dh, None
        return dh, dw


def lm_head_logits(h2d, weight):
    """[M, E] x [V, E]^T -> [M, V rounded up to a multiple of 64]; columns >= V are padding (see vocab_parallel_cross_entropy's
    `vocab_size`).  The usual GPT weight tying passes the embedding weight."""
    return _LMHeadFunction.apply(h2d, weight)


class _CrossEntropyFunction(torch.autograd.Function):
    """Forward: the per-token losses, one read of the logits.  Backward: the logits become their gradient, scaled, in one
    read and one write (the reference keeps its softmax in the logits' memory and scales it, :74, :97)."""

    @staticmethod
    def forward(ctx, logits, target, vocab_size):
        shape = target.shape
        l2 = logits.reshape(-1, logits.shape[-1])
        if not l2.is_contiguous():
            raise ValueError("vocab_parallel_cross_entropy overwrites its logits in place and needs them contiguous")
        flat = target.reshape(-1).contiguous()
        loss, stats = ops.cross_entropy_loss(l2, flat, vocab_size)
        # (the overwrite goes through the raw pointer: the logits are the output of a GEMM whose backward does not read
        # them)
        ctx.kept = l2.detach(), flat, stats, vocab_size
        ctx.lshape = logits.shape
        return loss.view(shape)

    @staticmethod
    def backward(ctx, grad_output):
        l2, flat, stats, vocab_size = ctx.kept
        scale = grad_output.reshape(-1).to(torch.float32).contiguous()
        if flat is None:            # a second backward: the logits are gone, their gradient is scaled once more
            ops.scale_rows_(l2, scale)
            return l2.view(ctx.lshape), None, None
        ctx.kept = l2, None, None, None
        return ops.cross_entropy_grad_(l2, flat, stats, scale, vocab_size).view(ctx.lshape), None, None


def vocab_parallel_cross_entropy(vocab_parallel_logits, target, vocab_size=None):
    """Per-token loss log(sum exp logits) - logits[target] (mpu/cross_entropy.py:109-110).  Like the reference's, its
    backward overwrites the logits (with their gradient).  vocab_size: number of valid leading columns when the logits
    come from lm_head_logits with a padded vocabulary."""
    V = vocab_parallel_logits.shape[-1] if vocab_size is None else vocab_size
    return _CrossEntropyFunction.apply(vocab_parallel_logits, target, V)
