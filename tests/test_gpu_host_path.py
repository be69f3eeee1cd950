"""The native host path of the operators (``dhellam_amd._host``): stream argument, results handed in, argument checks."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side", [False, True])
@pytest.mark.parametrize("tokens,hidden", [(1, 64), (33, 1000)])
def test_operators_on_a_stream_argument(side, tokens, hidden):
    """Results made on the given stream are those of the current stream, and ``profiling`` still reports a time."""
    from dhellam_amd.operators.layernorm import pylayernorm_bwd, pylayernorm_fwd
    from dhellam_amd.operators.swiglu import swiglu
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(tokens, hidden, generator=g, device="cuda")
    w = torch.randn(hidden, generator=g, device="cuda")
    st = torch.cuda.Stream() if side else None
    want = (torch.nn.functional.rms_norm(x, (hidden,), w, 1e-5), torch.nn.functional.silu(x[:, :hidden // 2]) * x[:, hidden // 2:])
    torch.cuda.synchronize()
    y, mu, rs, ms = pylayernorm_fwd(x, w, None, 1e-5, 0, False, st)
    assert mu is None and ms == 0
    a, ms = swiglu(x, st, profiling=True)
    assert ms > 0
    out = torch.empty_like(x)
    dx, dw, db, _ = pylayernorm_bwd(x, x, None, rs, w, 0, False, st, dgrad_out=out)
    assert dx.data_ptr() == out.data_ptr() and db is None and dw.shape == w.shape
    torch.cuda.synchronize()
    torch.testing.assert_close(y, want[0], rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(a, want[1], rtol=1e-5, atol=1e-5)


def test_argument_checks_keep_their_exceptions():
    from dhellam_amd.operators.bda import bda_fwd
    from dhellam_amd.operators.layernorm import pylayernorm_fwd
    from dhellam_amd.operators.rope import rope_fwd
    from dhellam_amd.operators.swiglu import swiglu
    x = torch.zeros(4, 6, device="cuda")
    with pytest.raises(AssertionError):
        swiglu(x[:, :5])                                                            # not contiguous, odd
    with pytest.raises(AssertionError):
        bda_fwd(x, x.half())
    with pytest.raises(AssertionError):
        pylayernorm_fwd(x, torch.ones(5, device="cuda"), None, 1e-5, 0, False, None)
    with pytest.raises(AssertionError):
        rope_fwd(x.view(4, 1, 6), x.view(4, 1, 6), torch.zeros(3, dtype=torch.int32, device="cuda"))
    with pytest.raises(RuntimeError, match="dtype"):
        swiglu(x.double())
