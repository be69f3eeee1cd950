"""Vocab-parallel cross entropy and the masked mean loss: dhellam/operators/loss.py:15-164.

Same calling convention as the reference (dict in, dict out, ``bwd(context, dout)``).  The
reference materialises the softmax in the forward and turns it into the gradient in the
backward; with ``keep_softmax=False`` the forward keeps only two numbers per row (maximum and
exponential sum) and the backward recomputes the softmax from the logits, which removes one
[rows, vocab] write and one read from the pair and leaves nothing of that size alive in
between.  ``output_dict["softmax"]`` is then None.

The all-reduces over the tensor-parallel group (loss.py:22-24,52-56,61-66) are the caller's:
with a world size above one the outputs are this rank's share.  The ranks join their row
statistics as

    M = max_r row_max_r,   S = sum_r sum_exp_r * exp(row_max_r - M),
    P = sum over the rank that holds the target of (predicted_r + row_max_r - M),
    loss = log S - P,

(two all-reduces of [rows] floats instead of the reference's three) and each rank's share of
the gradient comes from ``cross_entropy_bwd`` with ``row_max`` / ``sum_exp`` in its context
replaced by M / S (``keep_softmax=False``; a kept softmax is normalised by the rank's own sum).
"""
from __future__ import annotations

import torch

from .. import _host, _lib
from ..common.parallel_state import get_tensor_model_parallel_rank, get_tensor_model_parallel_world_size
from .embedding import vocab_range_from_per_partition_vocab_size


def cross_entropy_fwd(inputs, label_smoothing=0.0, keep_softmax=True):
    logits, target = inputs["vocab_parallel_logits"], inputs["target"]
    cols = logits.shape[-1]
    start, _ = vocab_range_from_per_partition_vocab_size(cols, get_tensor_model_parallel_rank(),
                                                        get_tensor_model_parallel_world_size())
    stats, softmax, mask, masked_target = _host.cross_entropy_fwd(logits, target, start, label_smoothing, keep_softmax)
    rows = mask.shape[0]
    if stats.shape[1] != rows:                         # no rows at all
        stats = stats[:, :rows]
    loss, row_max, sum_exp, predicted = stats.unbind(0)
    return {
        "loss": loss.view(target.shape),
        "label_smoothing": label_smoothing,
        "vocab_size": cols,
        "softmax": softmax.view(logits.shape) if keep_softmax else None,
        "target_mask": mask.view(target.shape),
        "masked_target_1d": masked_target,
        "row_max": row_max, "sum_exp": sum_exp, "predicted": predicted.view(target.shape),
    }


def cross_entropy_bwd(context, dout, grad_out=None):
    """Returns d loss / d logits scaled by ``dout`` per row.  With the softmax kept it is written
    over the softmax, as in the reference (loss.py:105-126); otherwise into ``grad_out`` (default:
    a new tensor; pass the logits themselves to overwrite them)."""
    inputs, out = context[0], context[1]
    logits, target = inputs["vocab_parallel_logits"], inputs["target"]
    cols = out["vocab_size"]
    start, _ = vocab_range_from_per_partition_vocab_size(cols, get_tensor_model_parallel_rank(),
                                                        get_tensor_model_parallel_world_size())
    if out["softmax"] is None:
        return _host.cross_entropy_bwd(logits, out["row_max"], out["sum_exp"], target, dout, start, out["label_smoothing"], grad_out)
    d = dout.to(torch.float32).contiguous()
    tgt = target.contiguous()
    rows = tgt.numel()
    assert d.numel() == rows
    sm = out["softmax"]
    s2 = sm.view(-1, cols)
    _lib.check(_lib.load().dh_cross_entropy_bwd(s2.data_ptr(), s2.stride(0), 0, None, None, tgt.data_ptr(), d.data_ptr(),
                                                rows, cols, start, float(out["label_smoothing"]), _lib.dt(sm),
                                                s2.data_ptr(), s2.stride(0), _host.stream_ptr(None)))
    return sm


def mask_scale_loss_fwd(inputs):
    """loss = sum(losses * mask) / sum(mask) / num_microbatch * loss_scale (loss.py:131-153).  The NaN
    assertion of the reference needs a host sync and is left to the caller."""
    scale = float(inputs["loss_scale"]) / float(inputs["num_microbatch"])
    out, m = _host.masked_mean_fwd(inputs["output_tensor"], inputs["loss_mask"], scale)
    return {"loss": out[0], "mask_sum": out[1:2], "mask_f32": m}


def mask_scale_loss_bwd(context, dout=None):
    """d loss / d output_tensor; like the reference (loss.py:155-164) the incoming gradient is one."""
    inputs, out = context[0], context[1]
    losses, m = inputs["output_tensor"], out["mask_f32"]
    scale = float(inputs["loss_scale"]) / float(inputs["num_microbatch"])
    return _host.masked_mean_bwd(m, out["mask_sum"], scale).view(losses.shape).to(losses.dtype)
