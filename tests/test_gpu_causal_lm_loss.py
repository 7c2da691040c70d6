"""FastForCausalLMLoss on 16-bit logits read in place, against the same function on the fp32 copy of them (which goes through
the general kernels): edges of the 16-byte chunks, odd vocabularies, rows that begin anywhere, ignored rows."""
import pytest
import torch

from tests.helpers import randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,s,V,offset", [(1, 2, 3, 0), (2, 9, 8, 8), (3, 5, 17, 1), (2, 7, 8195, 3), (2, 3, 32003, 0), (1, 4, 40960, 5)])
@pytest.mark.parametrize("shifted", [False, True])
def test_rows_in_place(b, s, V, offset, shifted, dtype):
    from fms_acceleration_foak.kernels.unsloth import FastForCausalLMLoss

    gen = torch.Generator().manual_seed(V)
    store = torch.empty(offset + b * s * V, dtype=dtype, device="cuda")
    store[offset:] = randn((b * s * V,), 5, dtype, scale=3.0).cuda()
    x = store[offset:].view(b, s, V)
    labels = torch.randint(0, V, (b, s), generator=gen)
    labels[:, 0] = labels[:, 1] = V - 1
    if s > 3:
        labels[b - 1, 2:4] = -100
        x[b - 1, 1 if not shifted else 2, V // 2] = float("inf")  # in a row without a label: not part of the loss
    labels = labels.cuda()
    kw = {"shift_labels": labels} if shifted else {}
    keep = x.clone()
    xa = x.detach().requires_grad_(True)
    la = FastForCausalLMLoss(xa, labels, V, **kw)
    (2.5 * la).backward()
    clean = torch.where(torch.isinf(keep), torch.zeros_like(keep), keep)  # the general backward multiplies such a row by zero
    xb = clean.float().requires_grad_(True)
    lb = FastForCausalLMLoss(xb * 1.0, labels, V, **kw)
    (2.5 * lb).backward()
    assert torch.equal(x, keep)  # the logits are left alone
    assert abs(la.item() - lb.item()) <= 2e-6 * max(1.0, abs(lb.item()))  # fp32 sums in another order
    # the gradients agree to fp32 rounding before their one rounding to the storage type: at most one unit apart
    ulp = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10
    tiny = 1e-30 if dtype == torch.bfloat16 else 2.0 ** -24
    diff = (xa.grad.float() - xb.grad).abs()
    assert bool((diff <= ulp * xb.grad.abs() + tiny).all())
    if not shifted:
        assert bool((xa.grad[:, -1] == 0).all())


def test_all_labels_ignored():
    from fms_acceleration_foak.kernels.unsloth import FastForCausalLMLoss

    x = randn((2, 5, 1000), 1, torch.bfloat16).cuda().requires_grad_(True)
    loss = FastForCausalLMLoss(x, torch.full((2, 5), -100, device="cuda"), 1000, num_items_in_batch=7)
    loss.backward()
    assert loss.item() == 0.0 and bool((x.grad == 0).all())


@pytest.mark.parametrize("shifted", [False, True])
def test_strided_labels(shifted):
    """Labels of one sequence that are a strided view: flattening them does not copy."""
    from fms_acceleration_foak.kernels.unsloth import FastForCausalLMLoss

    x = randn((1, 6, 100), 2, torch.bfloat16).cuda()
    labels = torch.arange(12, device="cuda").view(1, 12)[:, ::2]
    packed = labels.contiguous()
    kw = ({"shift_labels": labels}, {"shift_labels": packed}) if shifted else ({}, {})
    la, lb = FastForCausalLMLoss(x, labels, 100, **kw[0]), FastForCausalLMLoss(x, packed, 100, **kw[1])
    assert not labels.is_contiguous() and torch.equal(la, lb)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("V", [3, 17, 1024, 8195, 32003])
def test_a_nan_logit_stays(V, dtype):
    """One NaN anywhere in a row, also where a thread sees nothing finite before it: that row's loss and gradient are NaN
    and no other row's.  16-bit logits are read in place, fp32 ones by the general kernels (rows of whole chunks and not)."""
    import fmsa_hip

    columns = sorted({0, 1, V // 2, max(0, V - 9), V - 2, V - 1})
    x = randn((1, len(columns) + 1, V), V, dtype, scale=2.0).cuda()
    for row, c in enumerate(columns):
        x[0, row, c] = float("nan")
    labels = torch.full((len(columns) + 1,), V // 3, dtype=torch.int64, device="cuda")
    dloss = torch.ones(len(columns) + 1, device="cuda")
    if dtype == torch.float32:
        losses, lse = fmsa_hip.cross_entropy_fwd(x[0], labels)
        grad = fmsa_hip.cross_entropy_bwd_(x[0].clone(), dloss, lse, labels)
    else:
        losses, lse = fmsa_hip.cross_entropy_rows_fwd(x, labels, x.shape[1])
        grad = fmsa_hip.cross_entropy_rows_bwd(x, dloss, lse, labels, x.shape[1])[0]
    fused, fused_grad = fmsa_hip.cross_entropy_fused_(x[0].clone(), labels)
    for per_row in (losses, fused):
        assert bool(per_row[:-1].isnan().all()) and bool(per_row[-1].isfinite())
    for g in (grad, fused_grad):
        assert bool(g[:-1].isnan().all()) and bool(g[-1].isfinite().all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,s,V,offset", [(1, 3, 3, 1), (2, 9, 8, 0), (3, 5, 17, 1), (2, 7, 8195, 3), (2, 4, 40960, 0)])
@pytest.mark.parametrize("shifted", [False, True])
def test_logits_overwritten_before_the_backward(b, s, V, offset, shifted, dtype):
    """The gradient belongs to the logits the loss was taken of, whatever the caller writes over them afterwards."""
    from fms_acceleration_foak.kernels.unsloth import FastForCausalLMLoss

    store = torch.zeros(offset + b * s * V, dtype=dtype, device="cuda")
    store[offset:] = randn((b * s * V,), 7, dtype, scale=3.0).cuda()
    labels = torch.randint(0, V, (b, s), generator=torch.Generator().manual_seed(V)).cuda()
    labels[b - 1, s - 1] = -100
    kw = {"shift_labels": labels} if shifted else {}
    grads = []
    for overwrite in (False, True):
        leaf = store.clone().requires_grad_(True)
        x = (leaf * 1.0)[offset:].view(b, s, V)  # what a model hands over: not a leaf
        loss = FastForCausalLMLoss(x, labels, V, **kw)
        if overwrite:
            with torch.no_grad():
                x.mul_(0.5).add_(1.0)
        loss.backward()
        grads.append(leaf.grad)
    assert torch.equal(*grads) and bool((grads[0] != 0).any())
    with torch.no_grad():  # nothing is kept where no backward can follow
        assert torch.equal(FastForCausalLMLoss(store[offset:].view(b, s, V), labels, V, **kw), loss)


@pytest.mark.parametrize("rows,V", [(1, 16384), (3, 24579), (1500, 8192), (40, 16390)])
@pytest.mark.parametrize("mean", [True, False])
def test_parts_of_a_row_and_the_sum(rows, V, mean):
    """Rows cut into parts (chunks that do not divide evenly, ends on the first and last), more rows than the second launch has
    threads, labels read in place through their stride: against fp64."""
    import fmsa_hip

    x = randn((1, rows + 1, V), V, torch.bfloat16, scale=2.0).cuda()
    store = torch.randint(0, V, (2, 2 * rows + 2), generator=torch.Generator().manual_seed(rows)).cuda()
    labels = store[:1, : rows + 1]
    labels[0, 1::5] = -100
    if rows > 2:
        labels[0, 3] = V + 5  # no row of the loss, but counted as a label
    loss, (kept, lse, targets, count) = fmsa_hip.causal_lm_loss_fwd(x, labels[:, 1:], labels.stride(0), rows, mean, True)
    want = labels[0, 1:].clone()
    live = (want >= 0) & (want < V)
    exact = x[0, :rows].double()
    total = (exact.logsumexp(-1) - exact.gather(1, want.clamp(0, V - 1)[:, None])[:, 0])[live].sum()
    n = int((want != -100).sum()) if mean else 1
    assert torch.equal(targets, want) and count.item() == n
    # fp32: a sum of V exponentials each good to 1e-6, then a sum of the rows
    assert (n == 0 and loss.isnan()) or abs(loss.item() - total.item() / n) <= 1e-5 * max(1.0, abs(total.item() / n))
    labels.fill_(0)
    x.fill_(0)
    grad = fmsa_hip.causal_lm_loss_bwd(kept, lse, targets, count, torch.tensor(3.0, device="cuda"), rows)
    p = exact.softmax(-1)
    p[torch.arange(rows, device="cuda")[live], want[live]] -= 1.0
    ref = torch.where(live[:, None], p * (3.0 / max(n, 1)), torch.zeros_like(p))
    assert bool((grad[0, rows] == 0).all())
    assert bool(((grad[0, :rows].double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-9).all())


@pytest.mark.parametrize("rows", [8191, 8193])
def test_sum_of_more_rows_than_one_turn(rows):
    """Whole rows, whose losses the second launch takes 8192 a turn."""
    test_parts_of_a_row_and_the_sum(rows, 40, True)


def test_rows_by_themselves_are_those_of_the_sum():
    """cross_entropy_rows_fwd has no second launch; its losses add up to the call that has."""
    import fmsa_hip

    x, labels = randn((3, 41, 520), 5, torch.float16).cuda(), torch.randint(0, 520, (3, 41), generator=torch.Generator().manual_seed(6)).cuda()
    labels[1] = -100
    losses, lse = fmsa_hip.cross_entropy_rows_fwd(x, labels[:, 1:].reshape(-1).contiguous(), 40)
    loss, (_, lse2, _, count) = fmsa_hip.causal_lm_loss_fwd(x, labels[:, 1:], labels.stride(0), 40, False, True)
    assert torch.equal(lse, lse2) and bool((losses[40:80] == 0).all()) and count.item() == 1
    assert abs(losses.double().sum().item() - loss.item()) <= 120 * 2.0 ** -24 * losses.double().abs().sum().item()
