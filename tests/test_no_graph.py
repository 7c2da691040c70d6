"""When the fused operators run without an autograd node, and the autocast state their backward runs under."""
import pytest
import torch

from fms_acceleration_foak.autograd import bwd_as_fwd, no_graph, run


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


@pytest.mark.gpu
def test_backward_meets_the_autocast_state_of_its_forward():
    seen = []

    class F(torch.autograd.Function):
        @staticmethod
        @torch.amp.custom_fwd(device_type="cuda")
        def forward(ctx, x):
            return x.clone()

        @staticmethod
        @bwd_as_fwd
        def backward(ctx, dy):
            seen.append((torch.is_autocast_enabled("cuda"), torch.get_autocast_dtype("cuda")))
            return dy

    def state(dtype):
        return torch.autocast("cuda", dtype=dtype, enabled=dtype is not None)

    off = torch.get_autocast_dtype("cuda")
    for fwd in (None, torch.float16, torch.bfloat16):
        for bwd in (None, torch.float16, torch.bfloat16):
            x = torch.ones(2, device="cuda", requires_grad=True)
            with state(fwd):
                y = F.apply(x)
            with state(bwd):
                y.backward(torch.ones(2, device="cuda"))
            assert seen.pop()[0] is (fwd is not None)
            if fwd is not None:
                with state(bwd):
                    ctx = type("Ctx", (), {"_fwd_used_autocast": True, "_dtype": fwd})()
                    F.backward(ctx, torch.ones(2, device="cuda"))
                assert seen.pop() == (True, fwd)
    assert torch.get_autocast_dtype("cuda") == off
