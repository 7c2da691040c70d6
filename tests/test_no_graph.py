"""When the fused operators run without an autograd node: host-side rule, no GPU."""
import torch

from fms_acceleration_foak.autograd import no_graph, run


class _Double(torch.autograd.Function):
    nodes = 0

    @staticmethod
    def forward(ctx, x):
        ctx.save_for_backward(x)
        _Double.nodes += type(ctx).__name__ != "NoGraph"
        return 2 * x

    @staticmethod
    def backward(ctx, dy):
        return 2 * dy


def test_a_node_where_something_can_follow():
    x = torch.ones(3, requires_grad=True)
    assert not no_graph() and run(_Double, x).requires_grad and _Double.nodes == 1
    with torch.no_grad():
        assert no_graph() and not run(_Double, x).requires_grad and _Double.nodes == 1
        with torch.autograd.forward_ad.dual_level():
            assert not no_graph()
        seen = []
        torch.func.vmap(lambda y: seen.append(no_graph()) or y)(torch.ones(2, 3))
        assert seen == [False]
    with torch.inference_mode():
        assert no_graph()
