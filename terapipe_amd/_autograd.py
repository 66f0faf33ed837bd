"""What the autograd functions of the package ask the engine that runs their backward."""
import torch

from . import ops

_KNOWN = "terapipe_amd"     # in the metadata of an AccumulateGrad node: its _Leaf


class _Leaf:
    """What was seen of one AccumulateGrad node: the stream it runs on (None: it has not run yet) and where Python hooks on
    the node itself are kept."""
    __slots__ = ("stream", "pre", "post")

    def __init__(self, node):
        # The node's stream is that of the first forward that used the parameter while the graph was alive, which need
        # not be one of ours: it is read off when the node runs, by a hook that takes itself off again.
        self.stream = None

        def on_run(*_):
            self.stream = ops._stream()
            pre.remove()

        pre, post = node.register_prehook(on_run), node.register_hook(on_run)
        post.remove()
        self.pre, self.post = pre.hooks_dict_ref, post.hooks_dict_ref


def engine_adds_to_grad(ctx, params, first):
    """Whether the kernels of this node may add its gradients to the parameters' .grad (autograd gets None) in place of the
    engine.  ctx.next_functions[first:] are the parameters' AccumulateGrad nodes.  They have to run in the backward pass
    under way (under torch.autograd.grad they do not: the query raises for captured leaves), nobody may look at the
    gradients on the way (hooks on a parameter or on its node, a graph of the backward itself), and they have to run on
    THIS node's stream: what another node hands the engine for the same parameter is added there, and that stream is the
    one the caller of backward() waits for.  A node seen for the first time is only watched, so the first backward through
    a graph hands its gradients to the engine (which has nothing to add them to then, as a rule)."""
    if torch.is_grad_enabled():
        return False
    stream = ops._stream()
    ours = True
    try:
        for p, (node, _) in zip(params, ctx.next_functions[first:]):
            if getattr(node, "variable", None) is not p or not torch._C._will_engine_execute_node(node):
                return False
            known = node.metadata.get(_KNOWN)
            if known is None:
                node.metadata[_KNOWN] = _Leaf(node)
                ours = False
            elif known.stream != stream or known.pre() or known.post() or p._backward_hooks \
                    or getattr(p, "_post_accumulate_grad_hooks", None):
                ours = False
    except RuntimeError:
        return False
    return ours


def grad_to_add_to(ctx, param, first):
    """param.grad if the kernels may add to it in place of the engine (engine_adds_to_grad); otherwise None."""
    if not engine_adds_to_grad(ctx, (param,), first):
        return None
    g = param.grad
    if g is None or g.dtype != param.dtype or g.shape != param.shape or not g.is_contiguous() or g.is_sparse:
        return None
    return g
