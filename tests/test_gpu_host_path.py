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


@pytest.mark.parametrize("half", [False, True])
def test_attention_operands_off_the_gpu_are_refused(half):
    """Whole and half ring steps and the plain backward: an operand in host memory is an error, never an address that a
    kernel reads."""
    from dhellam_amd import _Clib
    from dhellam_amd.operators.ring_attn import RingGroup, fa_cp_block_bwd, fa_cp_block_fwd
    c, hq, hk, d = 32, 2, 1, 64
    g = torch.Generator(device="cuda").manual_seed(3)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    q, kv, cu = rand(1, 2, c, hq, d), [rand(2, 1, 2, c, hk, d) for _ in range(2)], torch.tensor([0, 2 * c], dtype=torch.int32, device="cuda")
    group, step, n = RingGroup(0, 2), int(half), 2 * c
    carry = fa_cp_block_fwd(q, cu, cu, n, n, kv, None, None, None, None, None, 0, True, group, [0, 1], None)[0]
    out, _, _, lse, rng = fa_cp_block_fwd(q, cu, cu, n, n, kv, *carry[2:7], 1, True, group, [0, 1], None)
    for at in range(4):
        a = [q, cu, cu, kv]
        a[at] = [t.cpu() for t in kv] if at == 3 else a[at].cpu()
        with pytest.raises((RuntimeError, AssertionError)):
            fa_cp_block_fwd(a[0], a[1], a[2], n, n, a[3], *([None] * 5 if step == 0 else carry[2:7]), step, True, group, [0, 1], None)
    for at in range(8):
        a = [rand(1, 2, c, hq, d), out, q, rand(1, 2, c, hq, d), lse, cu, cu, kv]
        a[at] = [t.cpu() for t in kv] if at == 7 else a[at].cpu()
        with pytest.raises((RuntimeError, AssertionError)):
            fa_cp_block_bwd(a[0], a[1], a[2], a[3], None, None, a[4], rng, a[5], a[6], n, n, a[7], 1 - step, True, group, [0, 1], None)
    x, s = [q.view(n, hq, d), kv[0][0].reshape(n, hk, d)], torch.empty(1, hq, n, device="cuda")
    args = [x[0], x[0], x[1], x[1], x[0], s, x[0].clone(), x[1].clone(), x[1].clone(), s.clone(), cu, cu]
    for at in range(len(args)):
        a = list(args)
        a[at] = a[at].cpu()
        with pytest.raises(RuntimeError):
            _Clib._attn_bwd_raw(*a, n, n, 0.1, True)


def test_data_gradient_results_of_another_shape_or_place_are_refused():
    """Few rows of a long reduction (the grouped kernel) refuse what the library product refuses."""
    from dhellam_amd._Clib import dgrad_gemm
    for n in (512, 8192):
        g, w = torch.ones(8, n, device="cuda", dtype=torch.bfloat16), torch.ones(n, 16, device="cuda", dtype=torch.bfloat16)
        assert torch.equal(dgrad_gemm(g, w, torch.empty(8, 16, device="cuda", dtype=torch.bfloat16)), torch.full((8, 16), float(n), device="cuda", dtype=torch.bfloat16))
        for bad in (torch.empty(16, 8, device="cuda", dtype=torch.bfloat16), torch.empty(8, 16, dtype=torch.bfloat16),
                    torch.empty(128, device="cuda", dtype=torch.bfloat16)):
            with pytest.raises(RuntimeError):
                dgrad_gemm(g, w, bad)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("t,n,k", [(1, 5120, 8), (256, 8192, 5120), (257, 7168, 4096), (512, 5120, 4096), (513, 5120, 4096), (1024, 8192, 3584),
                                   (1025, 5120, 512), (33, 5184, 136)])
def test_data_gradient_of_few_rows(t, n, k, dtype):
    """Both sides of the lines between the grouped kernel with one group (no table of offsets) and the library."""
    from dhellam_amd._Clib import dgrad_gemm
    from tests.util import assert_close
    g = torch.Generator(device="cuda").manual_seed(4)
    dy, w = (torch.randn(*s, generator=g, device="cuda").to(dtype) for s in ((t, n), (n, k)))
    assert_close(dgrad_gemm(dy, w), dy.double() @ w.double(), dtype, "dX")


@pytest.mark.parametrize("side", [False, True])
def test_zero_all(side):
    """More tensors than one launch takes, of all sizes and types, some of them not in the kernel's form; neighbours stay."""
    from dhellam_amd import _host
    sizes = [0, 4, 8, 20, 1000, 4096, 65540] + [12] * 60 + [1 << 20, 3]
    ts = [torch.full((n,), 7.0, device="cuda", dtype=[torch.float32, torch.bfloat16, torch.float16][i % 3]) for i, n in enumerate(sizes)]
    guard = torch.full((64, 64), 7.0, device="cuda")
    ts += [guard[:, :32], guard[40, 33:]]                    # a strided view, an address that is not a multiple of 16
    st = torch.cuda.Stream() if side else None
    if side:
        st.wait_stream(torch.cuda.current_stream())
    _host.zero_all(ts, st)
    torch.cuda.synchronize()
    assert all(torch.count_nonzero(t) == 0 for t in ts)
    assert (guard[:40, 32:] == 7).all() and (guard[41:, 32:] == 7).all() and guard[40, 32] == 7


def test_threads_on_one_stream_keep_their_scratch_apart():
    """Two threads issue operators of several kernels that hand each other data through the stream's scratch (split-k pieces,
    partial weight gradients): every result is that of one thread alone."""
    import threading
    from dhellam_amd.operators import moe
    from dhellam_amd.operators.layernorm import pylayernorm_bwd
    g = torch.Generator(device="cuda").manual_seed(6)
    jobs = []
    for i in range(2):
        a, b = torch.randn(40 + 8 * i, 4096, generator=g, device="cuda").bfloat16(), torch.randn(1, 256, 4096, generator=g, device="cuda").bfloat16()
        offs = torch.tensor([0, a.shape[0]], dtype=torch.int32, device="cuda")
        x, dy, w, rs = (torch.randn(*s, generator=g, device="cuda") for s in ((300, 2048), (300, 2048), (2048,), (300,)))
        jobs.append(lambda a=a, b=b, offs=offs, x=x, dy=dy, w=w, rs=rs: (moe.grouped_gemm_nt(a, b, offs),
                                                                        pylayernorm_bwd(dy, x, None, rs, w, 0, False, None)[1]))
    want = [job() for job in jobs]
    torch.cuda.synchronize()
    stream, got = torch.cuda.current_stream(), [[], []]

    def work(i):
        with torch.cuda.stream(stream):
            for _ in range(150):
                got[i].append(jobs[i]())
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for i in range(2):
        assert len(got[i]) == 150
        for c, dw in got[i]:
            assert torch.equal(c, want[i][0]) and torch.equal(dw, want[i][1])
