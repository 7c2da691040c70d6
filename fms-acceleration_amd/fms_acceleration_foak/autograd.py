"""Running the autograd functions of the fused operators: by themselves where no graph is built, and their backward under
the autocast state of their forward."""
import functools

import torch


class NoGraph:
    """Context of a pass that no backward follows: what is saved on it goes with it."""

    def save_for_backward(self, *tensors):
        pass


def no_graph() -> bool:
    """Whether a call can run its forward by itself, without an autograd node: no gradients are recorded, neither
    forward-mode AD nor a functorch transform (which would ask the autograd function for its rules) is active, and
    torch.jit is not tracing (the kernels are no torch operators: a graph that does not hold the autograd function holds
    the allocation of its outputs and nothing that fills them)."""
    return (not torch.is_grad_enabled() and torch.autograd.forward_ad._current_level < 0  # pylint: disable=protected-access
            and not torch._C._are_functorch_transforms_active()  # pylint: disable=protected-access
            and torch._C._get_tracing_state() is None)  # pylint: disable=protected-access


def run(function, *args):
    """function.apply(*args); without the node where nothing could follow from it."""
    return function.forward(NoGraph(), *args) if no_graph() else function.apply(*args)


def bwd_as_fwd(backward):
    """torch.amp.custom_bwd, whose autocast context costs the host 15 us a node, entered only where it would change
    something: where the state the backward meets is not the one its forward (torch.amp.custom_fwd) ran under."""
    entered = torch.amp.custom_bwd(backward, device_type="cuda")

    @functools.wraps(backward)
    def run_backward(ctx, *grads):
        on = torch.is_autocast_enabled("cuda")
        if on == ctx._fwd_used_autocast and (not on or torch.get_autocast_dtype("cuda") == ctx._dtype):  # pylint: disable=protected-access
            return backward(ctx, *grads)
        return entered(ctx, *grads)

    return run_backward
