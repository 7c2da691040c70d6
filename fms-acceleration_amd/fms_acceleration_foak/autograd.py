"""Running the autograd functions of the fused operators by themselves where no graph is built."""
import torch


class NoGraph:
    """Context of a pass that no backward follows: what is saved on it goes with it."""

    def save_for_backward(self, *tensors):
        pass


def no_graph() -> bool:
    """Whether a call can run its forward by itself, without an autograd node: no gradients are recorded, and neither
    forward-mode AD nor a functorch transform (which would ask the autograd function for its rules) is active."""
    return (not torch.is_grad_enabled() and torch.autograd.forward_ad._current_level < 0  # pylint: disable=protected-access
            and not torch._C._are_functorch_transforms_active())  # pylint: disable=protected-access


def run(function, *args):
    """function.apply(*args); without the node where nothing could follow from it."""
    return function.forward(NoGraph(), *args) if no_graph() else function.apply(*args)
