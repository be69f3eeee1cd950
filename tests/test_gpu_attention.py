"""GPU parity of flash attention (fwd, bwd), the merge and the ring step against the oracle.

All calls go through the C ABI via the reference-named shims (pymha_varlen_fwd/bwd,
fa_cp_block_fwd/bwd).  Inputs are seeded N(0,1), rounded to the run dtype and fed
identically to the HIP path and to the oracle.  Tolerances: rel-err <= 1e-2
(bf16/fp16), <= 1e-5 (fp32) on outputs and gradients.
"""
import math

import pytest
import torch

from oracle import attention as OA
from tests.util import assert_close, randn

pytestmark = pytest.mark.gpu


def _cu(lens):
    c = [0]
    for n in lens:
        c.append(c[-1] + n)
    return torch.tensor(c, dtype=torch.int32)


def _run_fwd_bwd(dtype, lens_q, lens_k, hq, hk, d, causal, oracle_dtype=torch.float64, packed=False, seed=0):
    from dhellam_amd import _Clib
    cq, ck = _cu(lens_q), _cu(lens_k)
    tq, tk = int(cq[-1]), int(ck[-1])
    scale = 1.0 / math.sqrt(d)
    if packed:
        # q, k, v as strided views of one [T, (hq + 2 hk) d] projection output (self-attention only)
        assert tq == tk
        qkv = randn((tq, (hq + 2 * hk) * d), dtype, seed)
        qkv_g = qkv.cuda()
        sl = lambda t, a, n: t[:, a * d:(a + n) * d].view(t.shape[0], n, d)
        q, k, v = sl(qkv, 0, hq), sl(qkv, hq, hk), sl(qkv, hq + hk, hk)
        qg, kg, vg = sl(qkv_g, 0, hq), sl(qkv_g, hq, hk), sl(qkv_g, hq + hk, hk)
    else:
        q, k, v = randn((tq, hq, d), dtype, seed), randn((tk, hk, d), dtype, seed + 1), randn((tk, hk, d), dtype, seed + 2)
        qg, kg, vg = q.cuda(), k.cuda(), v.cuda()
    do = randn((tq, hq, d), dtype, seed + 3)
    mq, mk = max(lens_q), max(lens_k)
    res = _Clib.pymha_varlen_fwd(qg, kg, vg, cq.cuda(), ck.cuda(), mq, mk, 0.0, scale, causal, False, 0, False)
    assert len(res) == 8
    out, lse = res[0], res[5]
    assert res[4] is out and res[1] is qg
    oo, lo = OA.attn_fwd(q, k, v, cq, ck, scale, causal, oracle_dtype)
    assert_close(out, oo, dtype, "out")
    for i, n in enumerate(lens_q):
        if n:
            assert_close(lse[i, :, :n], lo[i, :, :n], torch.float32, f"lse[{i}]")
    # backward consumes the forward's own (rounded) out and lse, like the layer does
    stream = torch.cuda.current_stream()
    r = _Clib.pymha_varlen_bwd(do.cuda(), qg, kg, vg, out, lse, cq.cuda(), ck.cuda(), mq, mk, 0.0, scale, causal,
                               None, False, 0, False, stream.cuda_stream)
    assert len(r) == 4
    dq, dk, dv, dl = r
    lse_cpu = lse.cpu().double()
    dqo, dko, dvo, dlo = OA.attn_bwd(do, q, k, v, out.cpu(), lse_cpu, cq, ck, scale, causal, oracle_dtype)
    assert_close(dq, dqo, dtype, "dq")
    assert_close(dk, dko, dtype, "dk")
    assert_close(dv, dvo, dtype, "dv")
    for i, n in enumerate(lens_q):
        if n:
            assert_close(dl[i, :, :n], dlo[i, :, :n], torch.float32, f"delta[{i}]")
    return out, lse, dq, dk, dv


def _fwd_path(lens_q, hq, d, causal):
    from dhellam_amd import _lib
    return _lib.load().dh_attn_fwd_path(len(lens_q), max(lens_q), sum(lens_q), hq, d, causal)


def _bwd_path(lens_q, lens_k, hq, hk, d, causal):
    from dhellam_amd import _lib
    lib, sizes = _lib.load(), (sum(lens_q), sum(lens_k))
    ws = lib.dh_attn_bwd_workspace_bytes(*sizes, len(lens_q), max(lens_q), hq, hk, d, _lib.DH_BF16)
    return lib.dh_attn_bwd_path(len(lens_q), max(lens_q), max(lens_k), *sizes, hq, hk, d, causal, ws)


@pytest.fixture(params=[True, False], ids=["keep_ds", "recompute"])
def ds_path(request):
    """Head dim 128 has two backward paths: dQ from the dS that the dK/dV pass keeps, or from recomputed S and dP."""
    from dhellam_amd import _Clib
    _Clib.set_attn_bwd_ds_limit(_Clib.ATTN_BWD_DS_LIMIT_DEFAULT if request.param else 0)
    yield request.param
    _Clib.set_attn_bwd_ds_limit()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens_q,lens_k,hq,hk,d,causal", [
    ([1024], [1024], 8, 1, 128, True),          # the 70B shard's head layout, shortened
    ([512, 512], [512, 512], 16, 16, 64, True),  # MHA, d 64, two sequences
    ([100, 257, 64, 1], [100, 257, 64, 1], 4, 2, 128, True),   # ragged
    ([300], [200], 4, 2, 128, False),            # rectangular, non-causal
    ([128, 77], [640, 33], 6, 3, 64, False),
    ([2048], [1024], 8, 2, 128, False),          # ring 'lower' shape
    ([1024], [2048], 8, 2, 128, False),          # ring 'upper' shape
    ([384, 129], [384, 129], 4, 4, 128, True),   # MHA at d 128: dK/dV written directly (no head split)
    ([128] * 4, [512] * 4, 64, 16, 128, False),  # many kv heads: two query heads per dK/dV workgroup
    ([0, 65, 33], [0, 65, 33], 4, 2, 128, True),   # an empty sequence in the batch
])
def test_attention_16bit(dtype, lens_q, lens_k, hq, hk, d, causal, ds_path):
    if d != 128 and not ds_path:
        pytest.skip("one backward path at this head dim")
    _run_fwd_bwd(dtype, lens_q, lens_k, hq, hk, d, causal)


@pytest.mark.parametrize("lens_q,lens_k,hq,hk,causal", [
    ([1024], [1024], 8, 1, True), ([300, 457, 64, 1], [300, 457, 64, 1], 24, 12, True), ([300, 40], [200, 97], 4, 2, False),
    ([2048], [1000], 8, 2, False),
])
def test_attention_backward_paths_agree(lens_q, lens_k, hq, hk, causal):
    """The two backward paths at head dim 128 on the same inputs: dV comes from the same kernel arithmetic
    (bit-identical); dK and dQ use delta = rowsum(dO * O), which the two paths sum in a different order (the delta
    kernel / the prologue of the recomputing dQ kernel), so a few of their elements differ in the last place."""
    from dhellam_amd import _Clib
    dtype, d = torch.bfloat16, 128
    cq, ck = _cu(lens_q).cuda(), _cu(lens_k).cuda()
    tq, tk, mq, mk = sum(lens_q), sum(lens_k), max(lens_q), max(lens_k)
    scale = 1.0 / math.sqrt(d)
    q, k, v, do = (randn((t, h, d), dtype, 30 + i).cuda() for i, (t, h) in enumerate(((tq, hq), (tk, hk), (tk, hk), (tq, hq))))
    res = _Clib.pymha_varlen_fwd(q, k, v, cq, ck, mq, mk, 0.0, scale, causal, False, 0, False)
    out, lse = res[0], res[5]
    sp = torch.cuda.current_stream().cuda_stream
    got = []
    try:
        for limit in (_Clib.ATTN_BWD_DS_LIMIT_DEFAULT, 0):
            _Clib.set_attn_bwd_ds_limit(limit)
            assert _bwd_path(lens_q, lens_k, hq, hk, d, causal) == (3 if limit else 5)      # else it is one path twice
            dq, dk, dv = torch.full_like(q, float("nan")), torch.full_like(k, float("nan")), torch.full_like(v, float("nan"))
            _Clib._attn_bwd_raw(do, q, k, v, out, lse, dq, dk, dv, None, cq, ck, mq, mk, scale, causal, sp)
            got.append((dq, dk, dv))
    finally:
        _Clib.set_attn_bwd_ds_limit()
    assert torch.equal(got[0][2], got[1][2])
    assert_close(got[0][1], got[1][1].double().cpu(), dtype, "dk of the two paths", scale=0.25)
    assert_close(got[0][0], got[1][0].double().cpu(), dtype, "dq of the two paths", scale=0.25)


def test_attention_packed_qkv_views():
    _run_fwd_bwd(torch.bfloat16, [384, 128], [384, 128], 8, 1, 128, True, packed=True)


def test_attention_full_70b_shard_shape():
    # 8 q heads + 1 kv head, d 128, 4096 tokens, causal, bf16; oracle in fp32 to keep the CPU time in seconds
    _run_fwd_bwd(torch.bfloat16, [4096], [4096], 8, 1, 128, True, oracle_dtype=torch.float32)


@pytest.mark.parametrize("lens_q,lens_k,hq,hk,d,causal", [
    ([512, 512], [512, 512], 16, 16, 64, True),  # the fp32 parity configuration
    ([130, 7], [130, 7], 4, 2, 32, True),
    ([50], [200], 2, 1, 256, False),
    ([70], [70], 3, 3, 20, True),
])
def test_attention_fp32(lens_q, lens_k, hq, hk, d, causal):
    _run_fwd_bwd(torch.float32, lens_q, lens_k, hq, hk, d, causal)


@pytest.mark.parametrize("dtype,hq,hk,d", [(torch.bfloat16, 4, 2, 128), (torch.float16, 32, 8, 128), (torch.bfloat16, 2, 2, 64),
                                         (torch.float32, 2, 1, 32)])
def test_attention_backward_accumulates_dq(dtype, hq, hk, d, ds_path):
    """dh_attn_bwd_acc with accumulate_dq: dq += the call's gradient (one rounding of the fp32 sum); dk, dv and a
    call without the flag are those of dh_attn_bwd."""
    from dhellam_amd import _Clib
    lens = [200, 56] if hq < 32 else [640]
    cu = _cu(lens).cuda()
    t, m, scale = sum(lens), max(lens), 1.0 / math.sqrt(d)
    q, k, v, do = (randn((t, h, d), dtype, 10 + i).cuda() for i, h in enumerate((hq, hk, hk, hq)))
    res = _Clib.pymha_varlen_fwd(q, k, v, cu, cu, m, m, 0.0, scale, True, False, 0, False)
    out, lse = res[0], res[5]
    sp = torch.cuda.current_stream().cuda_stream
    dq0, dk0, dv0 = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    _Clib._attn_bwd_raw(do, q, k, v, out, lse, dq0, dk0, dv0, None, cu, cu, m, m, scale, True, sp)
    base = randn((t, hq, d), dtype, 20).cuda()
    dq1, dk1, dv1 = base.clone(), torch.empty_like(k), torch.empty_like(v)
    _Clib._attn_bwd_raw(do, q, k, v, out, lse, dq1, dk1, dv1, None, cu, cu, m, m, scale, True, sp, accumulate_dq=True)
    assert torch.equal(dk1, dk0) and torch.equal(dv1, dv0)
    # the kernel adds its fp32 gradient before rounding, so it is at least as close to the exact sum as adding the
    # rounded gradient: compare with base + dq0 at the operator tolerance, and bit for bit where nothing was there
    assert_close(dq1, base.double().cpu() + dq0.double().cpu(), dtype, "dq accumulated")
    dq2 = torch.zeros_like(q)
    _Clib._attn_bwd_raw(do, q, k, v, out, lse, dq2, dk1, dv1, None, cu, cu, m, m, scale, True, sp, accumulate_dq=True)
    assert torch.equal(dq2, dq0)


def test_attention_is_deterministic():
    a = _run_fwd_bwd(torch.bfloat16, [700], [700], 8, 2, 128, True)
    b = _run_fwd_bwd(torch.bfloat16, [700], [700], 8, 2, 128, True)
    for x, y in zip(a, b):
        assert torch.equal(x, y)


def test_attention_profiling_and_errors():
    from dhellam_amd import _Clib
    q = randn((256, 4, 128), torch.bfloat16, 0).cuda()
    cu = _cu([256]).cuda()
    res = _Clib.pymha_varlen_fwd(q, q, q, cu, cu, 256, 256, 0.0, 0.1, True, False, 0, True)
    assert len(res) == 9 and res[8].device.type == "cpu" and res[8].item() > 0
    with pytest.raises(RuntimeError):
        _Clib.pymha_varlen_fwd(q, q, q, cu, cu, 256, 256, 0.1, 0.1, True, False, 0, False)   # dropout
    # the C ABI itself takes the compiled head dims only (the bindings pad other sizes before they call it)
    from dhellam_amd import _lib
    q72 = randn((256, 4, 72), torch.bfloat16, 0).cuda()
    o72, l72 = torch.empty_like(q72), torch.empty(1, 4, 256, device="cuda")
    rc = _lib.load().dh_attn_fwd(q72.data_ptr(), q72.data_ptr(), q72.data_ptr(), o72.data_ptr(), l72.data_ptr(),
                                 cu.data_ptr(), cu.data_ptr(), 1, 256, 256, 4, 4, 72, 288, 288, 288, 288, 0.1, 1,
                                 _lib.DH_BF16, torch.cuda.current_stream().cuda_stream)
    assert rc == -1 and "head dim" in _lib.load().dh_last_error().decode()
    k3 = randn((256, 3, 128), torch.bfloat16, 0).cuda()
    with pytest.raises(RuntimeError, match="multiple"):
        _Clib.pymha_varlen_fwd(q, k3, k3, cu, cu, 256, 256, 0.0, 0.1, True, False, 0, False)


# ------------------------------------------------------------------------------------------
# merge and ring step
# ------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_merge_kernel(dtype):
    from dhellam_amd import _Clib
    b, sq, hq, d = 2, 96, 3, 64
    row_begin, rows = [0, 0, 48, 48], [96, 96, 48, 48]
    outs = [randn((b * n, hq, d), dtype, 10 + i) for i, n in enumerate(rows)]
    lses = [randn((b, hq, n), torch.float32, 20 + i, std=3.0) for i, n in enumerate(rows)]
    out = torch.empty((b * sq, hq, d), dtype=dtype, device="cuda")
    lse = torch.empty((b, hq, sq), dtype=torch.float32, device="cuda")
    _Clib.pyattn_merge([o.cuda() for o in outs], [l.cuda() for l in lses], row_begin, rows, out, lse)
    oo, lo = OA.merge(outs, lses, row_begin, rows, b, sq, hq, d)
    assert_close(out, oo, dtype, "merged out")
    assert_close(lse, lo, torch.float32, "merged lse")


def _ring_inputs(dtype, b, c, hq, hk, d, cp, seed=0):
    q = randn((b, 2, c, hq, d), dtype, seed)
    chunks = [(randn((b, 2, c, hk, d), dtype, seed + 10 + 2 * i), randn((b, 2, c, hk, d), dtype, seed + 11 + 2 * i))
              for i in range(cp)]
    dout = randn((b, 2, c, hq, d), dtype, seed + 99)
    return q, chunks, dout


def _ring_gpu(q, chunks, dout, rank, cp):
    from dhellam_amd.operators.ring_attn import RingGroup, fa_cp_block_bwd, fa_cp_block_fwd
    b, _, c = q.shape[:3]
    s = 2 * c
    grp = RingGroup(rank, cp)
    cu = torch.arange(0, (b + 1) * s, s, dtype=torch.int32).cuda()
    bufs = [torch.stack((k, v)).cuda() for k, v in chunks]
    qg = q.cuda()
    carry = [qg, bufs, None, None, None, None, None, 0]
    for i in range(cp):
        r = fa_cp_block_fwd(carry[0], cu, cu, s, s, carry[1], carry[2], carry[3], carry[4], carry[5], carry[6], i,
                            True, grp, list(range(cp)), None)
        if i < cp - 1:
            carry, reqs = r
            assert reqs == [] and carry[-1] == i + 1
        else:
            out, q_ret, kv_ret, lse, rng = r
    assert q_ret is qg and kv_ret is bufs[-1]
    state = [dout.cuda(), None, None, bufs, 0]
    for i in range(cp + 1):
        r = fa_cp_block_bwd(state[0], out, qg, state[1], None, state[2], lse, rng, cu, cu, s, s, state[3], i, True,
                            grp, list(range(cp)), None)
        if i < cp:
            state, reqs = r
        else:
            dq, dkv = r
    return out, lse, dq, dkv


@pytest.mark.parametrize("dtype,b,c,hq,hk,d", [(torch.bfloat16, 1, 128, 4, 2, 128), (torch.bfloat16, 1, 96, 2, 2, 64),
                                                 (torch.float32, 1, 48, 2, 1, 32), (torch.bfloat16, 2, 64, 4, 2, 128)])
@pytest.mark.parametrize("rank", [0, 1, 3])
def test_ring_step_matches_oracle_and_dense(dtype, b, c, hq, hk, d, rank):
    cp = 4
    q, chunks, dout = _ring_inputs(dtype, b, c, hq, hk, d, cp)
    scale = 1.0 / math.sqrt(d)
    out, lse, dq, dkv = _ring_gpu(q, chunks, dout, rank, cp)
    oo, lo, _ = OA.ring_fwd(q, chunks, rank, scale)
    assert_close(out, oo, dtype, "ring out")
    assert_close(lse, lo, torch.float32, "ring lse")
    # the same thing as ONE dense causal attention over the zig-zag order
    do_, lo_ = OA.zigzag_dense(q, chunks, rank, scale)
    assert_close(out.view(b, 2 * c, hq, d), do_, dtype, "ring out vs dense")
    # backward: oracle ring with the GPU's own merged out/lse
    dqo, dkvo = OA.ring_bwd(dout, out.cpu(), lse.cpu().double(), q, chunks, rank, scale)
    assert_close(dq.view(q.shape), dqo, dtype, "ring dq")
    for s in range(cp):
        assert_close(dkv[s][0], dkvo[s][0], dtype, f"ring dk[{s}]")
        assert_close(dkv[s][1], dkvo[s][1], dtype, f"ring dv[{s}]")


@pytest.mark.parametrize("rank", [0, 1, 3])
def test_ring_step_full_size(rank):
    """The ring configuration at its full shape (q [1, 2, 2048, 32, 128], four visiting KV chunks of 8 kv heads;
    rank 0: a diagonal step and three half-q steps, rank 3: a diagonal step and three half-kv steps, rank 1:
    both kinds): forward and backward against ONE dense attention over the zig-zag positions, evaluated by the
    oracle in fp32 with its matmuls on the GPU (the [32, 4096, 16384] score tensor is 8.6 GB), gradients by
    autograd.  16-bit tolerance."""
    dtype, b, c, hq, hk, d, cp = torch.bfloat16, 1, 2048, 32, 8, 128, 4
    q, chunks, dout = _ring_inputs(dtype, b, c, hq, hk, d, cp, seed=3)
    scale = 1.0 / math.sqrt(d)
    out, lse, dq, dkv = _ring_gpu(q, chunks, dout, rank, cp)
    qr = q.cuda().float().requires_grad_()
    cr = [(k.cuda().float().requires_grad_(), v.cuda().float().requires_grad_()) for k, v in chunks]
    do_, lo_ = OA.zigzag_dense(qr, cr, rank, scale, dtype=torch.float32)
    assert_close(out.view(b, 2 * c, hq, d), do_, dtype, "ring out vs dense")
    assert_close(lse, lo_, torch.float32, "ring lse")
    (do_ * dout.cuda().float().view(b, 2 * c, hq, d)).sum().backward()
    assert_close(dq.view(q.shape), qr.grad, dtype, "ring dq")
    for s in range(cp):
        assert_close(dkv[s][0], cr[s][0].grad, dtype, f"ring dk[{s}]")
        assert_close(dkv[s][1], cr[s][1].grad, dtype, f"ring dv[{s}]")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d,lens,hq,hk,causal", [
    (96, [160, 37], 4, 2, True),            # compiled head dims beside 64 / 128 ...
    (192, [130, 64], 4, 1, True),
    (256, [96, 71], 2, 2, True),
    (256, [200], 4, 2, False),
    (80, [150, 33], 4, 2, True),            # ... and sizes that run zero-padded to the next one (the reference takes
    (40, [129], 2, 2, False),               # any d <= 256 and pads to a multiple of 8, flash_atten.cu:284,303-312)
    (160, [100, 90], 2, 1, True),
])
def test_attention_other_head_dims(dtype, d, lens, hq, hk, causal):
    """16-bit attention for head dims other than 64 / 128, forward and backward against the fp64 oracle, through
    the Python mirror of the binding and through the compiled extension (same bits)."""
    from dhellam_amd import _Clib
    import dhellam._Clib as C
    cu = _cu(lens)
    t, m = int(cu[-1]), max(lens)
    scale = 1.0 / math.sqrt(d)
    q, k, v, do = (randn((t, h, d), dtype, s) for s, h in ((0, hq), (1, hk), (2, hk), (3, hq)))
    qg, kg, vg, cug = q.cuda(), k.cuda(), v.cuda(), cu.cuda()
    res = _Clib.pymha_varlen_fwd(qg, kg, vg, cug, cug, m, m, 0.0, scale, causal, False, 0, False)
    out, lse = res[0], res[5]
    assert out.shape == q.shape
    d_run = res[4].shape[-1]
    assert d_run in _Clib.HEAD_DIMS_16BIT and d_run >= d and res[1].shape[-1] == d_run      # the "padded" slots
    oo, lo = OA.attn_fwd(q, k, v, cu, cu, scale, causal, torch.float64)
    assert_close(out, oo, dtype, "out")
    for i, n in enumerate(lens):
        assert_close(lse[i, :, :n], lo[i, :, :n], torch.float32, f"lse[{i}]")
    if d_run != d:
        assert torch.count_nonzero(res[4][..., d:]) == 0                                    # padding columns stay zero
    outc = out.contiguous()
    sp = torch.cuda.current_stream().cuda_stream
    dq, dk, dv, _ = _Clib.pymha_varlen_bwd(do.cuda(), qg, kg, vg, outc, lse, cug, cug, m, m, 0.0, scale, causal, None,
                                           False, 0, False, sp)
    assert dq.shape == q.shape and dk.shape == k.shape and dv.shape == v.shape
    dqo, dko, dvo, _ = OA.attn_bwd(do, q, k, v, outc.cpu(), lse.cpu().double(), cu, cu, scale, causal, torch.float64)
    assert_close(dq, dqo, dtype, "dq")
    assert_close(dk, dko, dtype, "dk")
    assert_close(dv, dvo, dtype, "dv")
    # the compiled extension pads and runs the same kernels
    rc = C.pymha_varlen_fwd(qg, kg, vg, cug, cug, m, m, 0.0, scale, causal, False, 0, False)
    assert torch.equal(rc[0], out) and rc[4].shape[-1] == d_run
    assert all(torch.equal(rc[5][i, :, :n], lse[i, :, :n]) for i, n in enumerate(lens))   # (entries past a sequence are not written)
    gc = C.pymha_varlen_bwd(do.cuda(), qg, kg, vg, outc, lse, cug, cug, m, m, 0.0, scale, causal, None, False, 0, False, sp)
    torch.cuda.synchronize()
    for a, b_ in zip(gc[:3], (dq, dk, dv)):
        assert torch.equal(a, b_)


def test_attention_head_dim_above_256_is_refused():
    from dhellam_amd import _Clib
    q = torch.zeros(8, 1, 264, dtype=torch.bfloat16, device="cuda")
    cu = _cu([8]).cuda()
    with pytest.raises(RuntimeError, match="256"):
        _Clib.pymha_varlen_fwd(q, q, q, cu, cu, 8, 8, 0.0, 1.0, True, False, 0, False)


@pytest.mark.parametrize("lens_q,lens_k,hq,hk,d,causal", [
    ([32, 1, 129], [32, 1, 129], 2, 1, 64, True),        # tile edges, one row, more tiles than wavefronts
    ([33], [160], 4, 2, 64, False), ([161, 31], [31, 64], 2, 2, 60, False),
    ([97], [97], 4, 1, 128, True), ([40], [300], 2, 2, 124, False), ([5], [5], 1, 1, 4, True),
])
def test_attention_f32_matrix_core_kernels(lens_q, lens_k, hq, hk, d, causal):
    """fp32 kernels for head dims up to 128: tile edges of both sequences, full and partial column tiles, GQA."""
    _run_fwd_bwd(torch.float32, lens_q, lens_k, hq, hk, d, causal)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens_q,lens_k,hq,hk,causal", [
    ([1, 33, 300], [1, 33, 300], 4, 2, True),            # tile edges, more sequences than one, longest last
    ([129], [129], 2, 1, True), ([70, 31], [257, 64], 2, 2, False), ([5], [3], 1, 1, False),
    ([1100], [1100], 64, 64, True),                      # the chip-filling form (128-row query tiles)
    ([520, 40], [200, 700], 64, 8, False),
])
def test_attention_head_dim_64(dtype, lens_q, lens_k, hq, hk, causal):
    """Head dim 64 kernels: both workgroup shapes, tile edges of both sequences, ragged batches, GQA groups."""
    _run_fwd_bwd(dtype, lens_q, lens_k, hq, hk, 64, causal)


@pytest.mark.parametrize("d", [64, 96])
def test_attention_backward_many_short_sequences_and_a_long_bound(d):
    """64 short sequences x 64 heads whose bound max_seqlen says 131072: the planes of the row statistics pass 2 GiB (they
    are laid out by the bound), the work does not.  Same gradients as with the bound at the longest length."""
    from dhellam_amd import _Clib
    dtype, lens, hq = torch.bfloat16, [1 + i % 7 for i in range(64)], 64
    cu = _cu(lens).cuda()
    t, scale = sum(lens), 1.0 / math.sqrt(d)
    q, k, v, do = (randn((t, hq, d), dtype, 40 + i).cuda() for i in range(4))
    got = []
    for m in (131072, max(lens)):
        res = _Clib.pymha_varlen_fwd(q, k, v, cu, cu, m, m, 0.0, scale, True, False, 0, False)
        got.append([res[0]] + _Clib.pymha_varlen_bwd(do, q, k, v, res[0], res[5], cu, cu, m, m, 0.0, scale, True, None, True, 0,
                                                     False, torch.cuda.current_stream().cuda_stream)[:3])
    # the bound picks the kernels' tile shapes, so sums may run in another order
    for a, b, what in zip(*got, ("out", "dq", "dk", "dv")):
        assert_close(a, b.double().cpu(), dtype, what)


# which kernels: forward 1 hand-ordered, 2 128-row tiles; backward 1 hand-ordered dK/dV, 2 dQ from kept dS or 4 hand-ordered dQ
# (8: with 128-row tiles); (with, without room for dS)
@pytest.mark.parametrize("lens_q,lens_k,hq,hk,causal,fwd,bwd", [
    ([512, 491], [512, 491], 64, 64, True, 3, (13, 13)),                # full rounds, rows that end inside a tile, MHA
    ([640, 300, 77, 513, 1, 200], [640, 300, 77, 513, 1, 200], 64, 8, True, 3, (13, 13)),     # several lengths, one row
    ([1537], [1537], 19, 19, True, 1, (3, 5)),                           # 64-row tiles
    ([300, 129], [200, 333], 16, 4, False, 1, (3, 5)),
    ([257, 100], [130, 31], 64, 16, False, 3, (13, 13)),
    ([100, 257, 64, 1], [100, 257, 64, 1], 48, 16, True, 2, (9, 9)),     # short rows, but many: dK/dV only
    ([0, 300, 65, 33], [0, 300, 65, 33], 48, 6, True, 2, (9, 9)),        # an empty sequence
    ([384, 129], [384, 129], 48, 48, True, 2, (3, 5)),                   # dK/dV of a head in one workgroup
    ([300, 200, 65], [300, 200, 65], 32, 4, True, 2, (3, 5)),
])
def test_attention_hand_ordered_kernels(lens_q, lens_k, hq, hk, causal, fwd, bwd, ds_path):
    """Head dim 128 on the kernels it has of its own, with ragged ends, empty sequences and split / unsplit GQA groups."""
    assert _fwd_path(lens_q, hq, 128, causal) == fwd
    assert _bwd_path(lens_q, lens_k, hq, hk, 128, causal) == bwd[not ds_path]
    _run_fwd_bwd(torch.bfloat16, lens_q, lens_k, hq, hk, 128, causal, oracle_dtype=torch.float32)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d,lens,hq,hk,causal,fwd,bwd", [
    (96, [257, 40, 1, 130], 64, 64, True, 2, 8), (96, [300, 33, 0, 96], 64, 16, False, 2, 8),
    (128, [257, 40, 1, 130], 64, 32, True, 2, 9),                # dQ and forward; dK/dV is the hand-ordered one here
    (192, [257, 33], 64, 64, True, 2, 0), (192, [130, 129], 80, 8, False, 2, 0),
    (256, [257, 33], 64, 32, True, 2, 0), (256, [130, 129], 80, 8, False, 2, 0),
])
def test_attention_chip_filling_tiles_of_other_head_dims(dtype, d, lens, hq, hk, causal, fwd, bwd):
    """The 128-row query tiles of the compiler-scheduled kernels, at the ends of tiles."""
    assert _fwd_path(lens, hq, d, causal) == fwd and _bwd_path(lens, lens, hq, hk, d, causal) == bwd
    _run_fwd_bwd(dtype, lens, lens, hq, hk, d, causal, oracle_dtype=torch.float32)


@pytest.mark.parametrize("d,lens_q,lens_k,hq,hk,causal,one", [
    (64, [28], [28], 3, 3, True, 1), (64, [65, 1, 0, 128], [65, 1, 0, 128], 4, 2, True, 1), (64, [40, 97], [200, 33], 8, 2, False, 1),
    (64, [512] * 2, [512] * 2, 16, 16, False, 0), (64, [1025], [1025], 32, 8, True, 1),          # both sides of the line
    (96, [33, 63], [33, 63], 4, 4, True, 1), (96, [200, 1], [64, 130], 4, 1, False, 1),
    (128, [31], [31], 2, 2, True, 1), (128, [100, 257, 64], [100, 257, 64], 4, 2, True, 1), (128, [70, 129], [70, 129], 8, 2, False, 1),
    (128, [7, 700], [7, 700], 4, 2, True, 1), (128, [801, 2, 324], [801, 2, 324], 8, 1, True, 0),     # one long among short
    (128, [1000] + [1] * 7, [1000] + [1] * 7, 8, 8, True, 1), (128, [3, 421, 5] + [2] * 13, [3, 421, 5] + [2] * 13, 8, 8, True, 1),
    (128, [599] + [1, 2] * 23, [599] + [1, 2] * 23, 4, 4, True, 0),     # ... of a grid for 128-row tiles
    (128, [224], [112], 4, 2, False, 1), (128, [97], [200], 6, 2, False, 1), (128, [300, 40], [200, 97], 4, 2, False, 0),
    (128, [44], [1300], 4, 2, False, 0), (128, [3], [600], 6, 2, False, 1), (128, [450], [675], 1, 1, False, 1),      # many keys
    (192, [97, 2], [97, 2], 4, 2, True, 1), (192, [65], [31], 2, 2, False, 1),
    (256, [129, 60], [129, 60], 2, 1, True, 1), (256, [32], [64], 4, 4, False, 1), (64, [50, 0], [20, 70], 2, 2, False, 1),
])
def test_attention_backward_in_one_launch(d, lens_q, lens_k, hq, hk, causal, one):
    """dK/dV and dQ by one grid behind the delta kernel: ragged ends, empty sequences, split and whole GQA groups,
    against the oracle; twice the same bits; delta zero past every sequence's end through the compiled module."""
    import importlib
    from dhellam_amd import _lib, _Clib
    t = sum(lens_q), sum(lens_k)
    assert _lib.load().dh_attn_bwd_one_launch(len(lens_q), max(lens_q), max(lens_k), *t, hq, hk, d, causal) == one
    _run_fwd_bwd(torch.bfloat16, lens_q, lens_k, hq, hk, d, causal, oracle_dtype=torch.float32)
    ext = importlib.import_module("dhellam._Clib")
    cq, ck = _cu(lens_q).cuda(), _cu(lens_k).cuda()
    q, k, v, do = (randn((n, h, d), torch.float16, 50 + i).cuda() for i, (n, h) in enumerate(zip((*t, t[1], t[0]), (hq, hk, hk, hq))))
    got = []
    for mod in (ext, ext, _Clib):
        junk = [torch.full((n,), float("nan"), device="cuda") for n in (2, 4, len(lens_q) * hq * max(lens_q))]
        del junk                                    # what the results are made in holds no zeros by chance
        res = mod.pymha_varlen_fwd(q, k, v, cq, ck, max(lens_q), max(lens_k), 0.0, d ** -0.5, causal, False, 0, False)
        assert res[7].tolist() == [0, 0]
        bwd = mod.pymha_varlen_bwd(do, q, k, v, res[0], res[5], cq, ck, max(lens_q), max(lens_k), 0.0, d ** -0.5, causal, res[7], True,
                                   0, False, torch.cuda.current_stream().cuda_stream)
        for i, n in enumerate(lens_q):
            assert (bwd[3][i, :, n:] == 0).all()
        got.append((res[0], *bwd))
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert torch.equal(a, b)


@pytest.mark.parametrize("d,lens,hq,hk,causal,dtype", [
    (128, [1537, 3], 19, 19, True, torch.bfloat16),              # dS kept: the delta kernel
    (128, [512, 491], 64, 64, True, torch.bfloat16),             # the hand-ordered dQ, paired tiles
    (128, [513, 70], 64, 64, False, torch.bfloat16),
    (64, [1100, 300], 64, 64, True, torch.bfloat16),             # the other dQ kernels
    (192, [300, 33, 257], 64, 64, True, torch.bfloat16), (64, [70, 33], 3, 3, True, torch.float32),
])
def test_attention_delta_is_zero_past_a_sequence(d, lens, hq, hk, causal, dtype):
    """Every kernel that writes delta as an output writes the rows past a sequence's end too."""
    from dhellam_amd import _Clib
    t, m, cu, scale = sum(lens), max(lens), _cu(lens).cuda(), d ** -0.5
    q, k, v, do = (randn((t, h, d), dtype, 60 + i).cuda() for i, h in enumerate((hq, hk, hk, hq)))
    out, lse = _Clib.pymha_varlen_fwd(q, k, v, cu, cu, m, m, 0.0, scale, causal, False, 0, False)[:6:5]
    want = (do.float() * out.float()).sum(-1)
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    delta = torch.full((len(lens), hq, m), float("nan"), device="cuda")
    _Clib._attn_bwd_raw(do, q, k, v, out, lse, dq, dk, dv, delta, cu, cu, m, m, scale, causal)
    # rowsum of d products in fp32: |error| <= d 2^-24 sum |dO O|
    bound = d * 2.0 ** -23 * (do.float() * out.float()).abs().sum(-1) + 1e-30
    at = 0
    for i, n in enumerate(lens):
        assert (delta[i, :, n:] == 0).all()
        assert ((delta[i, :, :n].t() - want[at:at + n]).abs() <= bound[at:at + n]).all()
        at += n


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens_q,lens_k,hq,hk,causal", [
    ([1001] * 4, [1001] * 4, 32, 8, True),                     # rows and keys that end inside a tile
    ([767] * 4, [37, 2, 640, 1], 32, 4, False),                   # fewer tiles of keys than stages
    ([1023, 300, 1, 77, 513, 255] * 2, [64, 1, 130, 33, 31, 95] * 2, 32, 32, False),
    ([600], [333], 32, 8, False),                              # 128-row tiles, two splits, an odd number of key tiles
    ([2689], [2689], 20, 4, True),
])
def test_attention_on_one_wavefront_a_simd(dtype, lens_q, lens_k, hq, hk, causal):
    """The kernels of 256- and 128-row query tiles (forward, recomputing dQ) at the edges of their tiles."""
    from dhellam_amd import _Clib
    assert _fwd_path(lens_q, hq, 128, causal) & 4
    _Clib.set_attn_bwd_ds_limit(0)
    try:
        _run_fwd_bwd(dtype, lens_q, lens_k, hq, hk, 128, causal, oracle_dtype=torch.float32)
    finally:
        _Clib.set_attn_bwd_ds_limit()


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("growth", [0.0, 12.0, -12.0])
def test_attention_forward_when_scores_grow_along_the_keys(causal, growth):
    """Scores that rise by many binades from key tile to key tile (the reference of the exponentials has to follow in some rows and
    not in others), that fall, and rows of nothing but equal scores."""
    from dhellam_amd import _Clib
    n, hq, d, dtype = 1024, 64, 128, torch.bfloat16
    assert _fwd_path([n, n], hq, d, causal) & 4
    q, k, v = (randn((2 * n, h, d), dtype, 60 + i) for i, h in enumerate((hq, 8, 8)))
    ramp = torch.linspace(0, abs(growth), n).repeat(2)
    k = ((ramp.flip(0) if growth < 0 else ramp) + 1)[:, None, None].mul(k.float()).to(dtype)
    q[::3] = 0
    cu, scale = _cu([n, n]), 1.0 / math.sqrt(d)
    res = _Clib.pymha_varlen_fwd(q.cuda(), k.cuda(), v.cuda(), cu.cuda(), cu.cuda(), n, n, 0.0, scale, causal, False, 0, False)
    oo, lo = OA.attn_fwd(q, k, v, cu, cu, scale, causal, torch.float32)
    assert_close(res[0], oo, dtype, "out")
    assert_close(res[5], lo, torch.float32, "lse")


def _bwd(do, q, k, v, out, lse, cq, ck, mq, mk, scale, causal):
    from dhellam_amd import _Clib
    return _Clib.pymha_varlen_bwd(do, q, k, v, out, lse, cq, ck, mq, mk, 0.0, scale, causal, None, True, 0, False,
                                  torch.cuda.current_stream().cuda_stream)[:3]


def _draw(dtype, lens_q, lens_k, hq, hk, seed):
    tq, tk = sum(lens_q), sum(lens_k)
    return [randn((t, h, 128), dtype, seed + i).cuda() for i, (t, h) in enumerate(((tq, hq), (tk, hk), (tk, hk), (tq, hq)))]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,m,hq,causal", [(2048, 256, 32, False), (1100, 352, 32, False), (512, 96, 8, False), (4096, 4096, 32, True), (2689, 2689, 40, True)])
def test_attention_with_a_scale_of_zero(dtype, n, m, hq, causal):
    """All scores equal: out and dV are means over the keys that a row sees, dQ and dK nothing.  (A mean of rounded values is off by
    half a unit of the last place at most, and so is a sum of products with weights that are rounded once.)"""
    from dhellam_amd import _Clib
    q, k, v, do = _draw(dtype, [n], [m], hq, 8, 80)
    cq, ck = _cu([n]).cuda(), _cu([m]).cuda()
    res = _Clib.pymha_varlen_fwd(q, k, v, cq, ck, n, m, 0.0, 0.0, causal, False, 0, False)
    keys = torch.arange(1, n + 1, device="cuda").double() if causal else torch.full((n,), float(m), device="cuda", dtype=torch.float64)
    mean = (v.double().cumsum(0) if causal else v.double().sum(0, keepdim=True)) / keys[:, None, None]
    assert_close(res[0], mean.repeat_interleave(hq // 8, 1).cpu(), dtype, "out")
    assert_close(res[5], keys.log().expand(1, hq, -1).cpu(), torch.float32, "lse")
    dq, dk, dv = _bwd(do, q, k, v, res[0], res[5], cq, ck, n, m, 0.0, causal)
    assert (dq == 0).all() and (dk == 0).all()
    part = (do.double() / keys[:, None, None]).view(n, 8, hq // 8, 128).sum(2)
    assert_close(dv, (part.flip(0).cumsum(0).flip(0) if causal else part.sum(0).expand(m, -1, -1)).cpu(), dtype, "dv")


# causal calls on each of the kernels with one wavefront a SIMD: 256-row tiles, 128-row tiles (two splits of the keys)
_CAUSAL_TILES = [([1024, 1001], 64, 8), ([2689], 20, 4), ([512, 491], 64, 64)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens,hq,hk", _CAUSAL_TILES[:2])
@pytest.mark.parametrize("key", [70, 335, 999])
def test_attention_forward_of_a_value_that_is_not_finite(dtype, lens, hq, hk, key):
    """A later key's V reaches no causal row outside its own block of 32: those rows stay what they are, bit for bit."""
    from dhellam_amd import _Clib
    assert _fwd_path(lens, hq, 128, True) & 4
    q, k, v, _ = _draw(dtype, lens, lens, hq, hk, 84)
    cu, n, scale = _cu(lens).cuda(), max(lens), 1.0 / math.sqrt(128)

    def run(v):
        r = _Clib.pymha_varlen_fwd(q, k, v, cu, cu, n, n, 0.0, scale, True, False, 0, False)
        return r[0], r[5]
    out, lse = run(v)
    first = key // 32 * 32
    for bad in (float("nan"), float("inf")):
        w = v.clone()
        w[key] = bad
        o2, l2 = run(w)
        assert torch.equal(o2[:first], out[:first]) and all(torch.equal(l2[i, :, :m], lse[i, :, :m]) for i, m in enumerate(lens))
        assert torch.equal(o2[lens[0]:], out[lens[0]:]) and not o2[key].isfinite().any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens,hq,hk", _CAUSAL_TILES)
@pytest.mark.parametrize("key", [70, 335, 480])
def test_attention_backward_of_keys_that_are_not_finite(dtype, lens, hq, hk, key):
    """A later key's K or V reaches no row of dQ outside its own block of 32."""
    from dhellam_amd import _Clib
    q, k, v, do = _draw(dtype, lens, lens, hq, hk, 88)
    cu, n, scale = _cu(lens).cuda(), max(lens), 1.0 / math.sqrt(128)
    r = _Clib.pymha_varlen_fwd(q, k, v, cu, cu, n, n, 0.0, scale, True, False, 0, False)
    first = key // 32 * 32
    _Clib.set_attn_bwd_ds_limit(0)
    try:
        dq = _bwd(do, q, k, v, r[0], r[5], cu, cu, n, n, scale, True)[0]
        for bad in (float("nan"), float("inf")):
            for which in range(2):
                kv = [k.clone(), v.clone()]
                kv[which][key] = bad
                dq2 = _bwd(do, q, *kv, r[0], r[5], cu, cu, n, n, scale, True)[0]
                assert torch.equal(dq2[:first], dq[:first]) and torch.equal(dq2[lens[0]:], dq[lens[0]:])
                assert dq2[key].isnan().any()
    finally:
        _Clib.set_attn_bwd_ds_limit()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens,hq,hk", [([1024, 1001], 64, 8), ([1537], 19, 19)])
@pytest.mark.parametrize("row", [5, 70, 671])
def test_attention_backward_of_rows_that_are_not_finite(dtype, lens, hq, hk, row, ds_path):
    """An earlier row's dO reaches no key of dK or dV outside its own block of 32."""
    from dhellam_amd import _Clib
    assert _bwd_path(lens, lens, hq, hk, 128, True) & 1
    q, k, v, do = _draw(dtype, lens, lens, hq, hk, 92)
    cu, n, scale = _cu(lens).cuda(), max(lens), 1.0 / math.sqrt(128)
    r = _Clib.pymha_varlen_fwd(q, k, v, cu, cu, n, n, 0.0, scale, True, False, 0, False)
    _, dk, dv = _bwd(do, q, k, v, r[0], r[5], cu, cu, n, n, scale, True)
    behind = row // 32 * 32 + 32
    for bad in (float("nan"), float("inf")):
        d2 = do.clone()
        d2[row] = bad
        _, dk2, dv2 = _bwd(d2, q, k, v, r[0], r[5], cu, cu, n, n, scale, True)
        assert torch.equal(dk2[behind:], dk[behind:]) and torch.equal(dv2[behind:], dv[behind:])
        assert not dv2[0].isfinite().all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,keys,hq,hk", [([800, 515], [960, 640], 48, 8), ([1537], [1600], 19, 19)])
def test_attention_backward_of_keys_that_no_row_sees(dtype, rows, keys, hq, hk, ds_path):
    """Causal, more keys than rows: what K holds behind the last row is met by nothing, also by the zeros that fill up the last tile
    of rows."""
    from dhellam_amd import _Clib
    assert _bwd_path(rows, keys, hq, hk, 128, True) & 1
    q, k, v, do = _draw(dtype, rows, keys, hq, hk, 96)
    cq, ck, mq, mk, scale = _cu(rows).cuda(), _cu(keys).cuda(), max(rows), max(keys), 1.0 / math.sqrt(128)
    r = _Clib.pymha_varlen_fwd(q, k, v, cq, ck, mq, mk, 0.0, scale, True, False, 0, False)
    clean = _bwd(do, q, k, v, r[0], r[5], cq, ck, mq, mk, scale, True)
    for bad in (float("nan"), float("-inf")):
        k2, at = k.clone(), 0
        for i, j in zip(rows, keys):
            k2[at + i:at + j] = bad
            at += j
        _, dk, dv = _bwd(do, q, k2, v, r[0], r[5], cq, ck, mq, mk, scale, True)
        assert torch.equal(dk, clean[1]) and torch.equal(dv, clean[2])


def _tiles(lens_q, lens_k, hq, hk, causal):
    """Query rows of a tile on one wavefront a SIMD (0: other kernels), forward and recomputing dQ."""
    from dhellam_amd import _lib
    lib, n, mq, mk, tq, tk = _lib.load(), len(lens_q), max(lens_q), max(lens_k), sum(lens_q), sum(lens_k)
    return (lib.dh_attn_fwd_rows(n, mq, mk, tq, hq, 128, causal),
            lib.dh_attn_bwd_dq_rows(n, mq, mk, tq, tk, hq, hk, 128, causal, 0))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens_q,lens_k,hq,hk,causal,fwd,dq", [
    ([2048], [333], 16, 8, False, 0, 128),                     # two splits of an odd number of key tiles
    ([1024, 1019], [333, 20], 16, 8, False, 0, 128),           # a second split without a key
    ([2000], [2000], 16, 16, False, 128, 128),
    ([700], [2000], 44, 44, False, 128, 128),                  # by the number of keys
    ([1100], [45], 32, 8, False, 0, 256),
    ([512, 491], [512, 491], 64, 64, True, 0, 128),
    ([961], [961], 64, 8, True, 0, 128),                       # odd numbers of tiles behind the diagonal
    ([600], [20], 32, 8, False, 128, 0),
    ([2689], [2689], 40, 8, True, 256, 256),
    ([767] * 4, [37, 2, 640, 1], 32, 4, False, 256, 256),
])
def test_attention_query_tiles_on_one_wavefront_a_simd(dtype, lens_q, lens_k, hq, hk, causal, fwd, dq):
    """Each form of the forward and of the recomputing dQ, at the ends of its tiles and splits."""
    from dhellam_amd import _Clib
    assert _tiles(lens_q, lens_k, hq, hk, causal) == (fwd, dq)
    _Clib.set_attn_bwd_ds_limit(0)
    try:
        _run_fwd_bwd(dtype, lens_q, lens_k, hq, hk, 128, causal, oracle_dtype=torch.float32)
    finally:
        _Clib.set_attn_bwd_ds_limit()


@pytest.mark.parametrize("lens_q,lens_k,hq,hk,tiles", [
    ([600, 600], [0, 333], 16, 4, (128, 0)), ([1024, 1019], [333, 0], 16, 8, (0, 128)),
    ([767] * 4, [37, 0, 640, 33], 32, 4, (256, 256)),
])
def test_attention_of_sequences_without_keys(lens_q, lens_k, hq, hk, tiles):
    """Rows that see nothing: out, dQ and delta are 0 and lse is -inf; the other sequences' results are those of a call without them."""
    from dhellam_amd import _Clib
    assert _tiles(lens_q, lens_k, hq, hk, False) == tiles
    q, k, v, do = _draw(torch.bfloat16, lens_q, lens_k, hq, hk, 100)
    cq, ck, mq, mk, scale = _cu(lens_q).cuda(), _cu(lens_k).cuda(), max(lens_q), max(lens_k), 1.0 / math.sqrt(128)
    _Clib.set_attn_bwd_ds_limit(0)
    try:
        r = _Clib.pymha_varlen_fwd(q, k, v, cq, ck, mq, mk, 0.0, scale, False, False, 0, False)
        dq, dk, dv = _bwd(do, q, k, v, r[0], r[5], cq, ck, mq, mk, scale, False)
    finally:
        _Clib.set_attn_bwd_ds_limit()
    aq = ak = 0
    for i, (n, m) in enumerate(zip(lens_q, lens_k)):
        sq, sk = slice(aq, aq + n), slice(ak, ak + m)
        if m == 0:
            assert (r[0][sq] == 0).all() and (dq[sq] == 0).all() and (r[5][i, :, :n] == float("-inf")).all()
        else:
            cpu = [t.cpu() for t in (do[sq], q[sq], k[sk], v[sk])]
            one = _cu([n]), _cu([m]), scale, False, torch.float32
            oo, lo = OA.attn_fwd(*cpu[1:], *one)
            want = OA.attn_bwd(*cpu, r[0][sq].cpu(), r[5][i:i + 1, :, :n].cpu().double(), *one)
            for got, ref, what in ((r[0][sq], oo, "out"), (dq[sq], want[0], "dq"), (dk[sk], want[1], "dk"), (dv[sk], want[2], "dv")):
                assert_close(got, ref, torch.bfloat16, what)
            assert_close(r[5][i, :, :n], lo[0], torch.float32, "lse")
        aq, ak = aq + n, ak + m


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens,hq,causal,rows", [([1100], 32, False, 128), ([2689], 20, True, 128), ([1024, 1001], 64, True, 256)])
@pytest.mark.parametrize("growth", [12.0, -12.0])
def test_attention_forward_when_scores_grow_in_every_form(dtype, lens, hq, causal, rows, growth):
    """The reference of the exponentials moves in both types, and in two splits of the keys each by itself."""
    from dhellam_amd import _Clib
    assert _tiles(lens, lens, hq, 4, causal)[0] == rows
    q, k, v, _ = (t.cpu() for t in _draw(dtype, lens, lens, hq, 4, 104))
    ramp = torch.cat([torch.linspace(0, abs(growth), n) for n in lens])
    k = ((ramp.flip(0) if growth < 0 else ramp) + 1)[:, None, None].mul(k.float()).to(dtype)
    q[::3] = 0
    cu, n, scale = _cu(lens), max(lens), 1.0 / math.sqrt(128)
    res = _Clib.pymha_varlen_fwd(q.cuda(), k.cuda(), v.cuda(), cu.cuda(), cu.cuda(), n, n, 0.0, scale, causal, False, 0, False)
    oo, lo = OA.attn_fwd(q, k, v, cu, cu, scale, causal, torch.float32)
    assert_close(res[0], oo, dtype, "out")
    for i, m in enumerate(lens):
        assert_close(res[5][i, :, :m], lo[i, :, :m], torch.float32, "lse")


@pytest.mark.parametrize("lens,hq,hk,causal,bound,tiles", [
    ([500 + i % 40 for i in range(65)], 8, 1, True, 540, (0, 256)),             # more sequences than are sorted
    ([800 + i % 5 for i in range(65)], 8, 2, False, 804, (256, 256)),
    ([100 + 7 * i for i in range(64)], 8, 8, True, 541, (0, 256)),              # as many as are
    ([300, 0, 513, 769, 64, 1, 700, 257], 40, 40, True, 769, (0, 256)),         # one head a kv head, an empty sequence
    ([785 - i for i in range(20)], 24, 8, True, 785, (256, 256)),               # odd numbers of tiles
    ([785 - i for i in range(20)], 20, 20, True, 785, (0, 256)),                # kv heads that go round the XCDs
    ([769 + i for i in range(12)], 40, 40, True, 780, (256, 256)),
    ([600 + i % 9 for i in range(24)], 24, 8, True, 608, (0, 128)),
    ([700, 300, 513, 1000, 640], 24, 8, False, 2048, (128, 256)),               # a bound that no sequence reaches
    ([257, 1100, 1, 300, 700, 700], 48, 16, False, 1100, (256, 256)),
])
def test_attention_workgroups_of_several_lengths(lens, hq, hk, causal, bound, tiles):
    """Every tile of every sequence and head is somebody's: kernels of one wavefront a SIMD count the workgroups that sequences have."""
    from dhellam_amd import _Clib, _lib
    lib, dtype, scale = _lib.load(), torch.bfloat16, 1.0 / math.sqrt(128)
    sizes = len(lens), bound, bound, sum(lens)
    assert (lib.dh_attn_fwd_rows(*sizes, hq, 128, causal), lib.dh_attn_bwd_dq_rows(*sizes, sum(lens), hq, hk, 128, causal, 0)) == tiles
    q, k, v, do = _draw(dtype, lens, lens, hq, hk, 108)
    cu = _cu(lens).cuda()
    _Clib.set_attn_bwd_ds_limit(0)
    try:
        r = _Clib.pymha_varlen_fwd(q, k, v, cu, cu, bound, bound, 0.0, scale, causal, False, 0, False)
        got = _Clib.pymha_varlen_bwd(do, q, k, v, r[0], r[5], cu, cu, bound, bound, 0.0, scale, causal, None, True, 0, False,
                                     torch.cuda.current_stream().cuda_stream)
    finally:
        _Clib.set_attn_bwd_ds_limit()
    cpu = [t.cpu() for t in (do, q, k, v)]
    oo, lo = OA.attn_fwd(*cpu[1:], cu.cpu(), cu.cpu(), scale, causal, torch.float32)
    lse = torch.full((len(lens), hq, max(lens)), float("-inf"), dtype=torch.float64)
    for i, n in enumerate(lens):
        lse[i, :, :n] = r[5][i, :, :n].cpu().double()
        assert_close(r[5][i, :, :n], lo[i, :, :n], torch.float32, "lse")
        assert (got[3][i, :, n:] == 0).all()
    want = OA.attn_bwd(*cpu, r[0].cpu(), lse, cu.cpu(), cu.cpu(), scale, causal, torch.float32)
    for a, b, what in zip([r[0], *got[:3]], [oo, *want[:3]], ("out", "dq", "dk", "dv")):
        assert_close(a, b, dtype, what)
