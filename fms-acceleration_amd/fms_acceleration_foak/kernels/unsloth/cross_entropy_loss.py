"""Cross-entropy loss on the gfx950 kernels of libfmsa_hip (drop-in for
kernels/unsloth/cross_entropy_loss.py of the reference: `Fast_CrossEntropyLoss` :195-262,
`fast_cross_entropy_loss` :265-282, `FastCrossEntropyLoss` :285-296, `FastForCausalLMLoss` :302-327,
`replace_custom_loss_when_triggered` :330-346).  As in the reference the backward overwrites the
saved logits with their gradient (:259), so a graph can be back-propagated once."""
from typing import Type

import torch

import fmsa_hip

from ...autograd import run


class Fast_CrossEntropyLoss(torch.autograd.Function):
    @staticmethod
    def forward(ctx, logits, labels):
        if logits.stride(1) != 1:
            logits = logits.contiguous()
        labels = labels.to(torch.int64).contiguous()
        losses, logsumexp = fmsa_hip.cross_entropy_fwd(logits, labels)
        ctx.save_for_backward(logits, logsumexp, labels)
        return losses

    @staticmethod
    def backward(ctx, dlosses):
        logits, logsumexp, labels = ctx.saved_tensors
        fmsa_hip.cross_entropy_bwd_(logits, dlosses.float(), logsumexp, labels)
        return logits, None, None


class Fast_CausalLMLossRows(torch.autograd.Function):
    """Sum (mean: over the labels that are not -100) of the losses of rows 0 .. seq_out - 1 of every sequence, read from the
    16-bit logits where they are; the gradient is a tensor of its own, so the logits stay as the caller sees them.  keep (a
    backward may follow): the forward leaves the rows it read and their labels in copies for the backward, so the caller may
    overwrite both before it, as with the fp32 copy of the general way."""

    @staticmethod
    def forward(ctx, logits, labels, label_stride, seq_out, mean, keep):
        loss, saved = fmsa_hip.causal_lm_loss_fwd(logits, labels, label_stride, seq_out, mean, keep)
        if keep:
            ctx.save_for_backward(*saved)
            ctx.seq_out = seq_out
        return loss

    @staticmethod
    def backward(ctx, dloss):
        return fmsa_hip.causal_lm_loss_bwd(*ctx.saved_tensors, dloss.float(), ctx.seq_out), None, None, None, None, None


def _rows_in_place(logits, labels, vocab_size, shifted):
    """Whether the loss can be taken from the logits as they are: 16-bit, contiguous [batch, seq, vocab] on the GPU, with a
    label per token (or per token after the shift).  Anything else goes the general way, through an fp32 copy."""
    return (logits.is_cuda and logits.dtype in (torch.float16, torch.bfloat16) and logits.dim() == 3 and logits.is_contiguous()
            and logits.shape[2] == vocab_size and 0 not in logits.shape and logits.shape[1] > (0 if shifted else 1)
            and (labels.numel() == logits.shape[0] * logits.shape[1] if shifted else labels.shape == logits.shape[:2])
            and not labels.is_floating_point())


def fast_cross_entropy_loss(logits, labels):
    """logits (batch, seq_len, vocab), labels (batch, seq_len) -> mean loss over labels != -100."""
    batch, seq_len, d = logits.shape
    assert labels.shape == (batch, seq_len)
    loss = Fast_CrossEntropyLoss.apply(logits.view(batch * seq_len, d), labels.view(-1))
    n_items = torch.count_nonzero(labels != -100)
    return loss.sum() / n_items


class FastCrossEntropyLoss(torch.nn.CrossEntropyLoss):
    def __init__(self):
        super().__init__()

    def forward(self, input, target):  # pylint: disable=redefined-builtin
        loss = Fast_CrossEntropyLoss.apply(input, target)
        n_items = torch.count_nonzero(target != -100)
        return loss.sum() / n_items


def FastForCausalLMLoss(logits, labels, vocab_size: int, num_items_in_batch: int = None, ignore_index: int = -100,
                        shift_labels=None, **kwargs):
    """Counterpart of transformers.loss.loss_utils.ForCausalLMLoss on the fused kernel."""
    if ignore_index == -100 and _rows_in_place(logits, labels if shift_labels is None else shift_labels, vocab_size, shift_labels is not None):
        # the fp32 copy, the shifted copy and their gradients' copies cost five times the two kernels
        seq_out = logits.shape[1] - (shift_labels is None)
        target = labels if shift_labels is None else shift_labels
        target = target.to(device=logits.device, dtype=torch.int64)
        if target.shape != logits.shape[:2] or target.stride(1) != 1:
            target = target.reshape(logits.shape[:2]).contiguous()
            if target.stride(1) != 1:  # (a single row of a strided view counts as contiguous)
                target = target.clone(memory_format=torch.contiguous_format)
        stride = target.stride(0)
        if shift_labels is None:
            target = target[:, 1:]  # the kernel reads the labels where they are, one token on
        loss = run(Fast_CausalLMLossRows, logits, target, stride, seq_out, num_items_in_batch is None,
                   torch.is_grad_enabled() and logits.requires_grad)
        return loss if num_items_in_batch is None else loss / num_items_in_batch
    logits = logits.float()
    if shift_labels is None:
        labels = labels.to(logits.device)
        shift_logits = logits[..., :-1, :].contiguous()
        shift_labels = labels[..., 1:].contiguous()
    else:  # newer transformers pass the labels already shifted, against the unshifted logits
        shift_logits = logits.contiguous()
    shift_logits = shift_logits.view(-1, vocab_size)
    shift_labels = shift_labels.reshape(-1).to(shift_logits.device)
    assert ignore_index == -100, "FastForCausalLMLoss currently supports only hardcoded ignore index -100."
    loss = Fast_CrossEntropyLoss.apply(shift_logits, shift_labels)
    if num_items_in_batch is not None:
        n_items = num_items_in_batch
    else:
        n_items = torch.count_nonzero(shift_labels != -100)
    return loss.sum() / n_items


def replace_custom_loss_when_triggered(module_cls: Type, custom_loss_type: str):
    """A trigger that performs the replacement itself: registers FastForCausalLMLoss under
    `custom_loss_type` in transformers' LOSS_MAPPING and points the model at it."""

    def _trigger(mod):
        if isinstance(mod, module_cls) and hasattr(mod, "loss_function"):
            from transformers.loss.loss_utils import LOSS_MAPPING  # pylint: disable=import-outside-toplevel

            LOSS_MAPPING[custom_loss_type] = FastForCausalLMLoss
            mod.loss_type = custom_loss_type
            return True
        return False

    return _trigger
