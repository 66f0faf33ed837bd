"""What the autograd functions of the package ask the engine that runs their backward."""
import weakref

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


_LOOKUPS = "terapipe_amd lookups"       # in the metadata of the node a weight's gradient goes to: see note_lookup
_TAKEN = object()


def note_lookup(node, index):
    """Remembers an autograd node whose backward adds a few rows to a dense gradient (an embedding): a product with the same
    weight may hand it that gradient (take_on).  node.next_functions[index] is the weight's."""
    weight, _ = node.next_functions[index]
    if weight is not None:
        node.stream, node.task, node.handed = ops._stream(), None, None
        seen = weight.metadata.setdefault(_LOOKUPS, [])
        seen[:] = [s for s in seen if s[0]() is not None] + [(weakref.ref(node), index)]


def lookup_to_hand_to(ctx, index):
    """A node (note_lookup) of the same weight, on the same stream, that is still to run in the backward pass under way, or
    None.  What it is handed becomes part of the one gradient it returns, so the engine sees the same sum as from two nodes:
    nothing of where that sum goes (.grad, a hook, torch.autograd.grad) is different."""
    weight = ctx.next_functions[index]
    if torch.is_grad_enabled() or weight[0] is None:
        return None
    task, stream = torch._C._current_graph_task_id(), ops._stream()
    for ref, at in weight[0].metadata.get(_LOOKUPS, ()):
        node = ref()
        if node is None or node.next_functions[at] != weight or node.stream != stream:
            continue
        if node.task != task:           # (what it was handed in a pass that broke off is dropped)
            try:
                if not torch._C._will_engine_execute_node(node):
                    continue
            except RuntimeError:
                continue
            node.task, node.handed = task, None
        if node.handed is not _TAKEN:
            return node
    return None


def taken_on(ctx):
    """In the backward of a node (note_lookup): the gradient it was handed, its own from now on, or None."""
    task = torch._C._current_graph_task_id()
    handed = ctx.handed if ctx.task == task else None
    ctx.task, ctx.handed = task, _TAKEN
    return handed
