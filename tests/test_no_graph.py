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


class _Opaque(torch.autograd.Function):
    """Fills its output behind torch's back, as the kernels do."""

    @staticmethod
    def forward(ctx, x):
        y = torch.empty_like(x)
        y.numpy()[...] = 3.0 * x.numpy()
        return y

    @staticmethod
    def backward(ctx, dy):
        return 3 * dy


def _traced(f, *args):
    """f under no_grad as torch.jit.trace records it, run on inputs of its own."""
    with torch.no_grad():
        return torch.jit.trace(f, tuple(torch.zeros_like(a) for a in args), check_trace=False)(*args)


def test_a_trace_holds_the_autograd_function():
    x = torch.arange(6.0).view(2, 3)
    assert torch.equal(_traced(lambda t: run(_Opaque, t), x), 3 * x)


def test_traces_of_the_norm_and_the_rotation(monkeypatch):
    """The operators that need no GPU to be entered, over stand-ins for their kernels."""
    import fmsa_hip
    from fms_acceleration_foak.kernels.unsloth import fast_rms_layernorm, fast_rope_embedding

    def norm(x, w, eps, gemma=False):
        y = torch.empty_like(x)
        y.numpy()[...] = 2.0 * x.numpy()
        return y, torch.empty(x.shape[0])

    def rotate(q, cos, sin, n_heads, head_dim, backward=False, strided=False):
        q.numpy()[...] *= -1.0
        return q

    def rotate_pair(q, k, cos, sin, head_dim):
        rotate(q, cos, sin, 0, head_dim)
        rotate(k, cos, sin, 0, head_dim)

    monkeypatch.setattr(fmsa_hip, "rms_layernorm_fwd", norm)
    monkeypatch.setattr(fmsa_hip, "rope_embedding_", rotate)
    monkeypatch.setattr(fmsa_hip, "rope_embedding_pair_", rotate_pair)
    layer = torch.nn.Module()
    layer.weight, layer.variance_epsilon = torch.nn.Parameter(torch.ones(8), requires_grad=False), 1e-5
    x = torch.randn(4, 8)
    assert torch.equal(_traced(lambda t: fast_rms_layernorm(layer, t), x), 2 * x)
    q, k, cos = torch.randn(1, 5, 4, 16), torch.randn(1, 5, 2, 16), torch.ones(5, 16)
    rotated = _traced(lambda a, b: fast_rope_embedding(a.clone().transpose(1, 2), b.clone().transpose(1, 2), cos, cos), q, k)
    for got, want in zip(rotated, (q, k)):
        assert torch.equal(got, -want.transpose(1, 2))


def test_one_launch_for_both_only_without_shared_storage(monkeypatch):
    """Two rotations of one memory have an order; two workgroups of one launch have none."""
    import fmsa_hip
    from fms_acceleration_foak.kernels.unsloth import fast_rope_embedding

    calls = []
    monkeypatch.setattr(fmsa_hip, "rope_embedding_", lambda q, *a, **k: calls.append(q.data_ptr()) or q)
    monkeypatch.setattr(fmsa_hip, "rope_embedding_pair_", lambda q, k, *a: calls.append("pair"))
    base, cos = torch.randn(192), torch.ones(2, 16)
    q = base[:128].view(1, 2, 4, 16).transpose(1, 2)
    with torch.no_grad():
        for k in (q, base[64:128].view(1, 2, 2, 16).transpose(1, 2), base[128:].view(1, 2, 2, 16).transpose(1, 2)):
            calls.clear()
            fast_rope_embedding(q, k, cos, cos)
            assert calls == [q.data_ptr(), k.data_ptr()]
        calls.clear()
        fast_rope_embedding(q, q.clone(memory_format=torch.preserve_format), cos, cos)
        assert calls == ["pair"]


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
