"""What the autograd functions of the package ask the engine that runs their backward."""
import weakref

import torch
from torch.utils.hooks import RemovableHandle

from . import ops

# In the metadata of an AccumulateGrad node: the stream it runs on, and how many handles of hooks had been made, on anything,
# when nobody had one on the node or on its parameter.
_KNOWN = "terapipe_amd"


def fresh_leaves(params):
    """Indices of the parameters that no autograd graph alive leads to, and that have no hooks: the next forward makes their
    AccumulateGrad nodes.  (Such a node holds its parameter: there is more than the Python object's reference to one that
    has a node.)  Where the first parameter has a node none is looked for: the kernels add all gradients of a node or none."""
    if params[0]._use_count() != 1:
        return ()
    return [i for i, p in enumerate(params) if p._use_count() == 1 and not _has_tensor_hooks(p)]


def _has_tensor_hooks(p):
    return bool(p._backward_hooks or getattr(p, "_post_accumulate_grad_hooks", None))


def note_leaves(node, first, fresh):
    """After a forward: what is known of the AccumulateGrad nodes that it made.  They run on the stream they were made on
    as long as they live, and nobody has put a hook on them yet.  node.next_functions[first:] are the parameters'."""
    if node is None or not fresh:
        return
    made = (ops._stream(), RemovableHandle.next_id)
    nodes = node.next_functions
    for i in fresh:
        leaf = nodes[first + i][0]
        if leaf is not None and leaf.metadata.setdefault(_KNOWN, made)[0] != made[0]:
            leaf.metadata[_KNOWN] = (None, 0)       # (two threads at once, on two streams)


def _has_hooks(node):
    """Python hooks on an autograd node, found by putting one beside them."""
    for register in (node.register_prehook, node.register_hook):
        handle = register(_has_hooks)
        n = len(handle.hooks_dict_ref())
        handle.remove()
        if n > 1:
            return True
    return False


def engine_adds_to_grad(ctx, params, first):
    """Whether the kernels of this node may add its gradients to the parameters' .grad (autograd gets None) in place of the
    engine.  ctx.next_functions[first:] are the parameters' AccumulateGrad nodes.  They have to run in the backward pass
    under way (under torch.autograd.grad they do not: the query raises for captured leaves), nobody may look at the
    gradients on the way (hooks on a parameter or on its node, a graph of the backward itself), and they have to be known
    to run on THIS node's stream (note_leaves): what another node hands the engine for the same parameter is added there,
    and that stream is the one the caller of backward() waits for.  A node that a forward of ours did not make -- somebody
    used the parameter first, or holds its node, as data-parallel wrappers do -- is not known."""
    if torch.is_grad_enabled():
        return False
    stream, handles = ops._stream(), RemovableHandle.next_id
    unsure = []
    try:
        for p, (node, _) in zip(params, ctx.next_functions[first:]):
            if getattr(node, "variable", None) is not p:
                return False
            known = node.metadata.get(_KNOWN)
            if known is None or known[0] != stream or not torch._C._will_engine_execute_node(node):
                return False
            if known[1] != handles:         # somebody has put a hook on something since
                unsure.append((p, node))
    except RuntimeError:
        return False
    if unsure:
        if any(_has_tensor_hooks(p) or _has_hooks(node) for p, node in unsure):
            return False
        for p, node in unsure:
            node.metadata[_KNOWN] = (stream, RemovableHandle.next_id)
    return True


_LOOKUPS = "terapipe_amd lookups"       # in the metadata of the node a weight's gradient goes to: see note_lookup
_TAKEN = object()


def note_lookup(node, index):
    """Remembers an autograd node whose backward adds a few rows to a dense gradient (an embedding): a product with the same
    weight may hand it that gradient (lookup_to_hand_to).  node.next_functions[index] is the weight's."""
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
    handed = ctx.handed if getattr(ctx, "task", None) == task else None
    ctx.task, ctx.handed = task, _TAKEN
    return handed
