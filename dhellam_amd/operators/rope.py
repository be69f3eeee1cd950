"""Rotary position embedding on q and k (rotate-half).

The reference has no RoPE; these wrappers follow its operator convention and sit
where a Llama layer needs them: after the q/k/v split and before the attention
call (dhellam/core/dstb.py:122-126), and on dq/dk before the dq|dk|dv concat in
backward (:376-382).
"""
from __future__ import annotations

import torch

from .. import _host
from ._util import issue

_inv_freq_cache: dict = {}


def rope_inv_freq(theta: float, d: int, device) -> torch.Tensor:
    """fp32 [d/2] table theta^(-2j/d), evaluated in double and rounded once."""
    key = (theta, d, device)
    t = _inv_freq_cache.get(key)
    if t is None:
        vals = [float(theta) ** (-2.0 * j / d) for j in range(d // 2)]
        t = torch.tensor(vals, dtype=torch.float64).to(torch.float32).to(device)
        _inv_freq_cache[key] = t
    return t


def _rope(q, k, positions, theta, seq_len, backward, stream, profiling, inplace):
    inv = rope_inv_freq(theta, q.shape[-1], q.device)
    (qo, ko), ms = issue(_host.rope, stream, profiling, q, k, inv, positions, int(seq_len or 0), backward, inplace)
    return (q, k, ms) if inplace else (qo, ko, ms)


def rope_fwd(q, k, positions=None, theta=10000.0, seq_len=None, stream=None, profiling=False, inplace=False):
    """q [tokens, hq, d], k [tokens, hk, d] (views with a token stride are fine).
    positions: int32 [tokens], or None for pos = t % seq_len (t if seq_len is None).
    Returns (q_rot, k_rot, ms)."""
    return _rope(q, k, positions, theta, seq_len, False, stream, profiling, inplace)


def rope_bwd(dq, dk, positions=None, theta=10000.0, seq_len=None, stream=None, profiling=False, inplace=False):
    """Gradient of rope_fwd: the inverse rotation applied to dq, dk."""
    return _rope(dq, dk, positions, theta, seq_len, True, stream, profiling, inplace)
