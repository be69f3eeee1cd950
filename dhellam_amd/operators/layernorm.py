"""Norm forward/backward with the reference's wrapper signatures.

Mirrors dhellam/operators/layernorm.py:6-45 (``pylayernorm_fwd``) and :47-91
(``pylayernorm_bwd``).  ``ln_bias=None`` selects RMSNorm (returned ``mu`` is
None); a bias selects LayerNorm.  ``fwd_sm_margin`` / ``bwd_sm_margin`` are
accepted and ignored (every reference call site passes 0, dstb.py:70,77,388).
"""
from __future__ import annotations

from .. import _host, _lib
from ._util import issue


def pylayernorm_fwd(inp, ln_weight, ln_bias, eps, fwd_sm_margin, zero_centered_gamma, stream, profiling=False,
                    residual=None, sum_out=None, ln_out=None):
    """Returns (ln_out, mu, rsigma, ms).  Extension over the reference signature: with ``residual`` the row that
    is normalised is ``inp + residual``, which is also stored in ``sum_out`` (default: a new tensor, returned
    as a fifth value) -- the reference's bda op and the norm after it (dstb.py:273-277, 73-78) in one pass.
    ``ln_out``: a contiguous tensor of the input's size to write the result into (e.g. this rank's rows of the
    buffer a sequence-parallel all-gather fills) instead of a new one."""
    if ln_out is not None:
        _lib.mark_written(ln_out)
    (y, mu, rsigma, total), ms = issue(_host.norm_fwd, stream, profiling, inp, ln_weight, ln_bias, eps,
                                       bool(zero_centered_gamma), residual, sum_out, ln_out)
    if residual is not None:
        return y, mu, rsigma, ms, total
    return y, mu, rsigma, ms


def pylayernorm_bwd(d_ln_out, inp, mu, rsigma, ln_weight, bwd_sm_margin, zero_centered_gamma, stream,
                    profiling=False, add_to_dgrad=None, dgamma_out=None, dbeta_out=None, dgrad_out=None):
    """Returns (dinp, dgamma, dbeta, ms).

    Extensions over the reference signature (all optional): ``add_to_dgrad`` is
    added to dinp inside the kernel (the residual-branch gradient the reference
    adds afterwards, dstb.py:391,401); ``dgamma_out`` / ``dbeta_out`` are
    accumulated into in place (the reference's ``main_grad.add_``, dstb.py:392-393);
    ``dgrad_out`` is a contiguous tensor of the input's size that receives dinp instead of a new one
    (``d_ln_out``, ``inp`` or ``add_to_dgrad`` itself, if that is not needed any more).
    """
    if dgrad_out is not None:
        _lib.mark_written(dgrad_out)
    (dinp, dgamma, dbeta), ms = issue(_host.norm_bwd, stream, profiling, d_ln_out, inp, mu, rsigma, ln_weight,
                                      bool(zero_centered_gamma), add_to_dgrad, dgamma_out, dbeta_out, dgrad_out)
    return dinp, dgamma, dbeta, ms
