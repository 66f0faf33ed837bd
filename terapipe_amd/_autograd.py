"""What the autograd functions of the package ask the engine that runs their backward."""
import torch


def engine_adds_to_grad(ctx, params, first):
    """Whether the backward pass under way is going to add this node's gradients to the parameters' .grad and nobody looks
    at them on the way: then the kernels can add them (and autograd gets None).  ctx.next_functions[first:] are the
    parameters' AccumulateGrad nodes; under torch.autograd.grad they do not run (the query raises for captured leaves),
    and a hook on a parameter or a graph of the backward itself (create_graph) needs the gradients as tensors."""
    if torch.is_grad_enabled():
        return False
    try:
        for p, (node, _) in zip(params, ctx.next_functions[first:]):
            if p._backward_hooks or getattr(p, "_post_accumulate_grad_hooks", None) or getattr(node, "variable", None) is not p \
                    or not torch._C._will_engine_execute_node(node):
                return False
    except RuntimeError:
        return False
    return True


def grad_to_add_to(ctx, param, first):
    """param.grad if the kernels may add to it in place of the engine (engine_adds_to_grad); otherwise None."""
    g = param.grad
    if g is None or g.dtype != param.dtype or g.shape != param.shape or not g.is_contiguous() or g.is_sparse:
        return None
    return g if engine_adds_to_grad(ctx, (param,), first) else None
