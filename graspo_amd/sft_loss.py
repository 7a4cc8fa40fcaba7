"""Drop-in for ``src/graspo/core/sft_loss.py``.

``sft_cross_entropy_loss`` is the mean token cross-entropy of the shifted
logits over the labels that are not ``ignore_index``, as
``F.cross_entropy(..., ignore_index=...)`` computes it in the reference
(sft_loss.py:12-34), without materialising the shifted copy or the [N, V]
softmax: the forward is the logprob kernel (one read of the logits), the
backward the logprob-gradient kernel (one read, one write).
"""

from __future__ import annotations

import torch

from . import ops


class _SFTCrossEntropy(torch.autograd.Function):
    @staticmethod
    def forward(ctx, logits, labels, ignore_index):
        # positions 0 .. S - 2 against labels 1 .. S - 1, both read in place
        out = ops.token_logprob(logits[:, :-1], labels[:, 1:], ignore_index=ignore_index,
                                mean=True)
        if out.bad_target:  # F.cross_entropy rejects a label outside [0, V)
            raise RuntimeError("sft_cross_entropy_loss: a label is outside [0, vocab_size)")
        # a copy of the targets (behind the rows, 8 bytes each): a loader may
        # refill its labels before the backward
        targets = labels[:, 1:].clone() if ctx.needs_input_grad[0] else None
        ctx.save_for_backward(logits, targets, out.logprob, out.count)
        ctx.ignore_index = ignore_index
        return out.mean_loss

    @staticmethod
    def backward(ctx, grad_loss):
        logits, targets, lp, count = ctx.saved_tensors
        grad = ops.token_logprob_backward(logits, targets, lp, grad_loss, mean_count=count,
                                          ignore_index=ctx.ignore_index)
        return grad, None, None


def sft_cross_entropy_loss(
    logits: torch.Tensor,
    labels: torch.Tensor,
    *,
    ignore_index: int = -100,
) -> torch.Tensor:
    """Mean cross-entropy of ``logits[:, :-1]`` against ``labels[:, 1:]``,
    skipping ``ignore_index`` (reference: sft_loss.py:12-34).  ``logits`` is
    [B, S, V] in fp32, bf16 or fp16; the loss is an fp32 scalar."""
    if logits.dim() != 3 or labels.shape != logits.shape[:2]:
        raise ValueError(
            f"expected logits [B, S, V] and labels [B, S], got {tuple(logits.shape)} and "
            f"{tuple(labels.shape)}")
    if logits.stride(-1) != 1:
        logits = logits.contiguous()
    return _SFTCrossEntropy.apply(logits, labels, int(ignore_index))
