"""Fused-head counterpart of the reference's SFT `chunked_nll` loss
(`_chunked_cross_entropy_loss`, trl/trainer/sft_trainer.py:117-234)."""
from __future__ import annotations

import math

import torch
from torch import Tensor

from .utils import _masked_head

__all__ = ["_chunked_cross_entropy_loss"]


def _chunked_cross_entropy_loss(
    hidden_states: Tensor,
    lm_head_weight: Tensor,
    chunk_size: int,
    labels: Tensor | None = None,
    shift_labels: Tensor | None = None,
    num_items_in_batch: Tensor | int | None = None,
    logit_scale: float = 1.0,
    final_logit_softcapping: float | None = None,
    lm_head_bias: Tensor | None = None,
) -> tuple[Tensor, Tensor, Tensor, Tensor]:
    """Next-token cross-entropy over hidden states and an `lm_head` weight without materialising logits.

    Same arguments and return value as the reference: `(loss, correct_count, entropy_sum, n_valid)` over the
    local batch; `labels` are shifted here, `shift_labels` are taken as already aligned; `-100` positions are
    dropped before the matmul; the loss is `sum / num_items_in_batch` if that is given, else the mean over
    valid tokens.  `chunk_size` is the number of vocabulary rows that the backward takes at a time where memory is
    short: it is raised to what 1 GiB of workspace holds where that much can be allocated (the reference chunks tokens;
    the kernels need no token chunking).  `correct_count` counts tokens whose label holds the row maximum."""
    if labels is None and shift_labels is None:
        raise ValueError("At least one of `labels` or `shift_labels` must be provided.")
    h = hidden_states.shape[-1]
    shifted = shift_labels is None and labels.shape == hidden_states.shape[:-1]
    if shifted:  # label t + 1 belongs to position t; the last position has none
        shape = math.prod(labels.shape[:-1]), labels.shape[-1]
        hidden, targets = hidden_states.reshape(*shape, h), labels.reshape(shape)[:, 1:]
    elif shift_labels is not None:
        hidden, targets = hidden_states.reshape(1, -1, h), shift_labels.reshape(1, -1)
    else:  # (labels of another shape that leave one label per remaining position)
        hidden, targets = hidden_states[..., :-1, :].reshape(1, -1, h), labels[..., 1:].reshape(1, -1)
    # what the loss is divided by, where the head's own function can do it
    mean_of = "count"
    if isinstance(num_items_in_batch, Tensor):
        mean_of = None
        if (num_items_in_batch.dim() == 0 and num_items_in_batch.dtype in (torch.int64, torch.int32, torch.float32)
                and not num_items_in_batch.requires_grad):
            mean_of = num_items_in_batch.to(device=hidden.device, dtype=torch.float32)
    elif num_items_in_batch is not None:
        mean_of = num_items_in_batch if type(num_items_in_batch) in (int, float) else None
    try:
        logp, ent, hit, n_valid = _masked_head(hidden, lm_head_weight, targets, targets, 1.0, chunk_size,
                                               final_logit_softcapping, logit_scale, lm_head_bias, -100, True, False, shifted,
                                               mean_of)
    except (ValueError, TypeError, NotImplementedError):
        if bool((targets != -100).any()):
            raise
        logp, n_valid = targets.new_empty(0), targets.new_zeros((), dtype=torch.int64)  # nothing enters the head
    if logp.numel() == 0:
        # whole micro-batch masked: keep the loss attached to every trainable input (sft_trainer.py:186-195)
        loss = (hidden_states.float().sum() + lm_head_weight.float().sum()) * 0.0
        if lm_head_bias is not None:
            loss = loss + lm_head_bias.float().sum() * 0.0
        zero = hidden.new_zeros((), dtype=torch.float32)
        return loss, zero, zero.clone(), n_valid
    if mean_of is not None:
        return logp, hit, ent, n_valid
    loss = -logp.sum()
    if num_items_in_batch is None:
        loss = loss / n_valid
    else:
        if isinstance(num_items_in_batch, Tensor):
            num_items_in_batch = num_items_in_batch.to(loss.device)
        loss = loss / num_items_in_batch
    return loss, hit.sum(), ent.sum(), n_valid
