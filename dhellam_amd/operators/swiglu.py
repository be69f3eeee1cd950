"""SwiGLU forward/backward: dhellam/operators/swiglu.py:28-62.

``y`` has the gate in the first half of the last dim and the up projection in
the second half (swiglu.py:15).
"""
from __future__ import annotations

from .. import _host, _lib
from ._util import issue


def swiglu(y, stream=None, profiling=False, with_transposed=False):
    """``with_transposed``: the kernel also writes the result transposed ([f, rows], for the weight-gradient product
    of the projection behind the activation) and hangs it on the returned tensor, where ``_Clib.wgrad_gemm`` finds
    it; ignored for shapes or types the kernel does not take."""
    (out, ot), ms = issue(_host.swiglu_fwd, stream, profiling, y, with_transposed)
    if ot is not None:
        out._dh_rows_transposed = (out._version, ot)        # valid while nothing has written ``out`` since
    return out, ms


def swiglu_back(g, y, o=None, stream=None, profiling=False, with_transposed=False):
    """``o`` (optional) receives the result; the reference allocates it but its kernel
    ignores it (swiglu.py:48-55).  ``with_transposed``: the kernel also writes the result transposed
    ([2f, rows], for the weight-gradient product of the projection in front of the activation) and hangs it on the
    returned tensor, where ``_Clib.wgrad_gemm`` finds it; ignored for shapes or types the kernel does not take."""
    (out, ot), ms = issue(_host.swiglu_bwd, stream, profiling, g, y, o, with_transposed)
    if o is not None:
        _lib.mark_written(o)                # a reused ``o`` may carry the transposed twin of an earlier call
    if ot is not None:
        out._dh_rows_transposed = (out._version, ot)        # valid while nothing has written ``out`` since
    return out, ms
