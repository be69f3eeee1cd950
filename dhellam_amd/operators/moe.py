"""MoE routing, token permute/unpermute and the grouped expert FFN for one
expert-parallel rank.

The reference has no MoE; these operators follow its wrapper convention
(``stream=None`` means the current stream, trailing elapsed-ms return) and the
dropless top-k semantics of Mixtral / Megatron-core.  All row counts stay on the
device (``MoEPlan.expert_offsets``): nothing here synchronises with the host, so
buffers are sized by the caller-provided ``max_rows`` bound.
"""
from __future__ import annotations

from dataclasses import dataclass

import torch

from .. import _host
from .._Clib import _note_read, transposed_of
from ._util import issue


@dataclass
class MoEPlan:
    """Result of sorting the flat (token, slot) assignment list by expert."""
    tokens: int
    k: int
    num_experts: int
    tokens_per_expert: torch.Tensor   # int32 [E]
    expert_offsets: torch.Tensor      # int32 [E + 1]
    sorted_idx: torch.Tensor          # int32 [T * k], assignment ids in sorted order
    dest_row: torch.Tensor            # int32 [T * k], sorted position of each assignment


def route_topk(logits, k, stream=None, profiling=False):
    """logits fp32 [T, E] -> (topk_idx int32 [T, k], gates fp32 [T, k], ms).  Descending
    logit, ties to the lower expert id; gates = softmax over the k selected logits."""
    (idx, gates), ms = issue(_host.moe_route, stream, profiling, logits, k)
    return idx, gates, ms


def sort_assignments(topk_idx, num_experts, stream=None, profiling=False):
    """Stable counting sort of the assignments by expert id -> (MoEPlan, ms)."""
    (tpe, offs, order, dest), ms = issue(_host.moe_sort, stream, profiling, topk_idx, num_experts)
    return MoEPlan(topk_idx.shape[0], topk_idx.shape[1], num_experts, tpe, offs, order, dest), ms


def _gather(x, plan, e_lo, e_hi, max_rows, row_scale, stream, profiling):
    return issue(_host.moe_gather, stream, profiling, x, plan.sorted_idx, row_scale, plan.expert_offsets, e_lo, e_hi,
                 max_rows, plan.k)


def _scatter(y, plan, e_lo, e_hi, gates, stream, profiling):
    return issue(_host.moe_scatter, stream, profiling, y, plan.dest_row, gates, plan.expert_offsets, e_lo, e_hi,
                 plan.tokens, plan.k)


def permute_fwd(x, plan, e_lo, e_hi, max_rows, stream=None, profiling=False):
    """x [T, H] -> (permuted [max_rows, H], ms): the rows routed to local experts
    [e_lo, e_hi), grouped by expert, original (token, slot) order inside an expert.
    Rows past the real count are zero."""
    return _gather(x, plan, e_lo, e_hi, max_rows, None, stream, profiling)


def permute_bwd(d_permuted, plan, e_lo, e_hi, stream=None, profiling=False):
    """Gradient of permute_fwd: dx[t] = sum of the local rows that came from token t."""
    return _scatter(d_permuted, plan, e_lo, e_hi, None, stream, profiling)


def unpermute_fwd(y, plan, gates, e_lo, e_hi, stream=None, profiling=False):
    """y [rows, H] (expert outputs, permuted order), gates fp32 [T, k] ->
    (out [T, H], ms) with out[t] = sum_j gates[t, j] * y[row(t, j)] over local assignments."""
    assert gates.dtype == torch.float32 and gates.is_contiguous()
    return _scatter(y, plan, e_lo, e_hi, gates, stream, profiling)


def unpermute_bwd(dout, y, plan, gates, e_lo, e_hi, max_rows, stream=None, profiling=False):
    """Returns (dy [max_rows, H], dgates fp32 [T, k], ms): dy[r] = gate * dout[token(r)],
    dgates[t, j] = <dout[t], y[row(t, j)]> (0 for assignments owned by other ranks)."""
    (dy, dgates), ms = issue(_host.moe_unpermute_bwd, stream, profiling, dout, y, plan.sorted_idx, plan.dest_row, gates,
                             plan.expert_offsets, e_lo, e_hi, max_rows, plan.tokens, plan.k)
    return dy, dgates, ms


# ---------------------------------------------------------------------------------------
# grouped GEMM and the expert FFN built from it
# ---------------------------------------------------------------------------------------
def grouped_gemm_nt(a, b, offs, max_rows=None, out=None, stream=None):
    """c[rows_g] = a[rows_g] @ b[g].T ; a [R, K], b [G, N, K] -> c [R, N]."""
    return _host.grouped_gemm(a, b, offs, max_rows, out, True, stream)


def grouped_gemm_nn(a, b, offs, max_rows=None, out=None, stream=None):
    """c[rows_g] = a[rows_g] @ b[g] ; a [R, K], b [G, K, N] -> c [R, N]."""
    return _host.grouped_gemm(a, b, offs, max_rows, out, False, stream)


def grouped_gemm_tn(a, b, offs, out=None, accumulate=False, stream=None):
    """c[g] (+)= a[rows_g].T @ b[rows_g] ; a [R, M], b [R, N] -> c [G, M, N]."""
    return _host.grouped_gemm_tn(a, b, offs, out, accumulate, stream)


def expert_ffn_fwd(xp, w1, w2, offs, stream=None, profiling=False):
    """SwiGLU FFN of the local experts on permuted rows.  xp [R, H]; w1 [G, 2F, H] (gate |
    up); w2 [G, H, F]; offs int32 [G + 1] (a slice of MoEPlan.expert_offsets).
    Returns (y [R, H], (h, a) saved for backward, ms)."""
    (y, h, a), ms = issue(_host.expert_ffn_fwd, stream, profiling, xp, w1, w2, offs)
    return y, (h, a), ms


def expert_ffn_bwd(dy, xp, w1, w2, offs, saved, dw1=None, dw2=None, stream=None, profiling=False):
    """Backward of expert_ffn_fwd.  Returns (dxp, dw1, dw2, ms); dw1/dw2 are accumulated
    into when given (the reference accumulates weight gradients into main_grad,
    dhellam/core/dstb.py:547-592)."""
    h, a = saved

    def ffn(st):
        # data gradients: against the resident transposes of the expert weights where the caller keeps them
        # (``_Clib.keep_transposed``): the same products in the forward's layout, which the grouped kernel runs faster
        w2t, w1t = transposed_of(w2, st), transposed_of(w1, st)
        res = _host.expert_ffn_bwd(dy, xp, w1, w2, w1t, w2t, offs, h, a, dw1, dw2, st)
        if w1t is not None or w2t is not None:
            _note_read(w2, st)
            _note_read(w1, st)
        return res
    (dxp, g1, g2), ms = issue(ffn, stream, profiling)
    return dxp, g1, g2, ms
