"""Build-time checks that need no GPU."""
import re
import shutil

import pytest


needs_hipcc = pytest.mark.skipif(shutil.which("hipcc") is None and not __import__("os").path.exists("/opt/rocm/bin/hipcc"),
                                 reason="needs hipcc")


@needs_hipcc
def test_grouped_gemm_loads_are_left_alone_until_used():
    """The chip-filling grouped GEMM copies its operands to LDS from assembly and orders reads, waits, copies and barriers
    by hand: the compiled loop has to keep that order, without spills, in all of the ten instantiations (NT / NN with and
    without the split last round, TN; bf16 and fp16).  ``check_grouped_gemm_loops`` compiles the source to assembly and
    verifies that; a violation raises."""
    from dhellam_amd.build import check_grouped_gemm_loops
    assert check_grouped_gemm_loops() == 10


@pytest.fixture(scope="module")
def gemm_kernels():
    from dhellam_amd.build import grouped_gemm_assembly
    return grouped_gemm_assembly()


@needs_hipcc
@pytest.mark.parametrize("where", ["before the loop", "main loop", "last slice", "behind it"])
def test_grouped_gemm_check_covers_the_first_and_the_last_slices(gemm_kernels, where):
    """A counted wait that is missing anywhere on the way is found: in front of the main loop, in it, in the separately compiled
    slice of an odd number, and the last wait before LDS is used again."""
    from dhellam_amd.build import check_grouped_gemm_order
    for fn in gemm_kernels:
        counted = [i for i, l in enumerate(fn) if l.strip() == "s_waitcnt vmcnt(8)"]
        assert len(counted) == 1 + 6 + 3
        last = next(i for i in range(counted[-1], len(fn)) if fn[i].strip().startswith("s_waitcnt vmcnt(0)"))
        bad = list(fn)
        bad[{"before the loop": counted[0], "main loop": counted[3], "last slice": counted[8], "behind it": last}[where]] = ""
        with pytest.raises(RuntimeError):
            check_grouped_gemm_order(bad)


def test_weight_gradients_of_very_long_rows_stay_with_the_library():
    """The grouped kernel's tiles address rows of fewer than 2^22 elements."""
    from dhellam_amd import _host
    edge = (1 << 22) - 8
    assert _host.wgrad_grouped(16, edge, 256) and _host.wgrad_grouped(16, 256, edge)
    assert not _host.wgrad_grouped(16, edge + 8, 256) and not _host.wgrad_grouped(16, 256, edge + 8)
    assert not _host.wgrad_grouped(16, 5000000, 256)


@pytest.mark.parametrize("dtype,rows,cols,one", [
    (1, 16, 8, 1), (1, 64, 64, 1), (1, 512, 512, 1), (1, 1024, 1024, 1), (1, 1280, 4096, 1), (1, 512, 8192, 1),
    (1, 64, 8, 0), (1, 768, 64, 0), (1, 256, 128, 0), (1, 768, 256, 0), (1, 1024, 512, 0), (1, 1025, 1024, 0), (1, 2048, 8192, 0),
    (0, 48, 8, 1), (0, 512, 256, 1), (0, 768, 384, 1), (0, 1024, 1024, 1), (0, 1280, 2048, 1), (0, 256, 64, 0), (0, 768, 256, 0)])
def test_norm_backward_in_one_launch_is_for_rows_that_few_workgroups_can_take(dtype, rows, cols, one):
    """The one launch has a workgroup per 32 columns: with few columns it is the faster form for few rows only."""
    from dhellam_amd import _lib
    assert _lib.load().dh_norm_bwd_one_launch(rows, cols, dtype) == one


@pytest.mark.parametrize("t,n,k,grouped", [
    # measured the faster one here, on both sides of every line
    (1000, 32000, 1024, 1), (16384, 16032, 4096, 1), (8, 16000, 256, 1), (1000, 8192, 1024, 1), (65, 8192, 1024, 1), (64, 5120, 256, 1),
    (200, 12288, 256, 1), (8192, 7168, 8192, 1), (8, 5120, 4096, 1), (16384, 1000, 64, 1), (8192, 1256, 1024, 1), (32, 1504, 512, 1),
    (1000, 1504, 128, 1), (64, 2008, 1024, 1), (1000, 4008, 256, 1), (256, 6008, 128, 1), (6000, 8192, 64, 1), (12000, 8192, 128, 1),
    # ... and by the library
    (16384, 8192, 64, 0), (16384, 8192, 128, 0), (16384, 32000, 64, 0), (256, 5120, 256, 0), (48, 8192, 1024, 0), (63, 5120, 256, 0),
    (1000, 1256, 1024, 0), (8, 1256, 1024, 0), (8192, 1504, 512, 0), (1000, 2008, 1024, 0), (128, 4008, 256, 0), (3000, 8192, 2048, 0),
    (1000, 3072, 1024, 0), (1904, 1280, 8192, 0), (16, (1 << 22), 256, 0)])
def test_data_gradients_go_where_they_were_measured_the_faster(t, n, k, grouped):
    from dhellam_amd import _host
    assert _host.dgrad_grouped(t, n, k) == bool(grouped)


@pytest.mark.parametrize("t,n,k,grouped", [
    (24, 100000, 8, 1), (1000, 8, 100000, 1), (4096, 100000, 8, 0), (32, 32, 100000, 1), (1000, 100000, 32, 1),
    (1000, 50304, 64, 1), (2000, 50304, 64, 0), (8192, 64, 65536, 0), (1000, 50304, 96, 1), (2000, 50304, 96, 0), (1000, 128, 50304, 1),
    (2000, 128, 50304, 0), (3000, 264, 30000, 1), (4096, 30000, 264, 0), (8192, 320, 65536, 0), (2000, 192, 50304, 1), (8192, 512, 50304, 1),
    (4096, 7168, 8192, 1), (4096, 8192, 3584, 1), (4096, 1280, 8192, 0), (1000, 1280, 8192, 1), (384, 32000, 96, 1), (385, 1280, 2048, 0)])
def test_weight_gradients_go_where_they_were_measured_the_faster(t, n, k, grouped):
    from dhellam_amd import _host
    assert _host.wgrad_grouped(t, n, k) == bool(grouped)


@pytest.mark.parametrize("groups,rows,m,n,accumulate,tiles", [
    (16, 256, 5632, 4096, 1, 256), (1, 16, 4096, 4096, 1, 256), (32, 64, 1304, 136, 1, 256), (8, 2048, 5632, 1024, 0, 128),
    (8, 16384, 5632, 4096, 0, 256), (16, 1600, 5632, 4096, 0, 128), (1, 4096, 8192, 1024, 1, 128),
    # most of a 256-wide tile past the matrix
    (32, 64, 5552, 8, 1, 128), (64, 6400, 16, 4112, 1, 128), (16, 4465, 32, 10704, 1, 128), (64, 1446, 1056, 80, 1, 128),
    # rows past the 32-bit offsets of a tile's old values
    (1, 16, 256, 4300800, 1, 0), (1, 16, 4300800, 256, 1, 0), (1, 16, 256, (1 << 22) - 8, 1, 256)])
def test_tiles_of_a_grouped_weight_gradient(groups, rows, m, n, accumulate, tiles):
    from dhellam_amd import _lib
    assert _lib.load().dh_grouped_gemm_tn_tiles(groups, rows, m, n, accumulate) == tiles


@pytest.mark.parametrize("tokens,experts,k,lanes", [
    (1, 1, 1, 1), (64, 2, 2, 1), (100, 3, 3, 8), (1000, 5, 4, 8), (8192, 8, 2, 8), (65536, 8, 2, 1), (131072, 8, 8, 1), (16384, 16, 4, 16),
    (65536, 16, 2, 1), (8192, 24, 2, 32), (65536, 24, 2, 1), (16384, 64, 8, 64), (65536, 64, 1, 1), (131072, 64, 8, 64), (262144, 48, 1, 1)])
def test_lanes_of_the_routing(tokens, experts, k, lanes):
    """A scan where it was measured the faster: few experts, or tokens enough to fill the chip with a thread each."""
    from dhellam_amd import _lib
    assert _lib.load().dh_moe_route_lanes(tokens, experts, k) == lanes


@pytest.mark.parametrize("rows,cols,k,form,own", [
    (1024, 5632, 1024, "TN", 1), (1024, 2816, 1024, "TN", 1), (777, 2816, 1024, "TN", 0), (1024, 1536, 1024, "TN", 0), (1024, 4000, 2048, "TN", 0),
    (1024, 16032, 1024, "TN", 0), (1024, 2816, 1000, "TN", 0), (1000, 5568, 256, "NN", 1), (1024, 2816, 1023, "NN", 0), (1024, 2818, 1024, "NN", 0),
    (5632, 1024, 1024, "NT", 1), (5632, 1024, 1001, "NT", 1), (1024, 1024, 1024, "NT", 0), (512, 512, 64, "NT", 1), (4, 4, 1, "NT", 1),
    (514, 512, 64, "NT", 0), (512, 514, 64, "NT", 0), (512, 512, 193, "NT", 0), (4352, 768, 227, "NT", 0), (1 << 21, 8, 64, "NT", 0)])
def test_fp32_products_go_where_they_were_measured_the_faster(rows, cols, k, form, own):
    """D [rows, cols]; what the copies cannot take (lengths that are no multiples of 16 bytes) is the library's."""
    from dhellam_amd import _lib
    assert _lib.load().dh_gemm_f32_path(cols, rows, k, form[0] == "T", form[1] == "T") == own


@pytest.mark.parametrize("rows,k,own", [(5632, 1280, 1), (5632, 1281, 0), (2816, 1536, 1), (2816, 1537, 0)])
def test_fp32_weight_gradients_of_two_rounds_end_sooner(rows, k, own):
    """[rows, 1024] of k rows: 1408 and 704 tiles of 64 x 64."""
    from dhellam_amd import _lib
    assert _lib.load().dh_gemm_f32_path(1024, rows, k, 0, 1) == own


@pytest.fixture(scope="module")
def loops():
    import importlib.util
    from dhellam_amd.build import CSRC
    spec = importlib.util.spec_from_file_location("attn_loops", CSRC / "attn_loops.py")
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def test_attention_loops_keep_their_own_account(loops):
    """The attention loops are written with an account of what is in flight; every form of them passes it."""
    assert loops.generate().count("#define DH_") >= 5


@pytest.mark.parametrize("fault,code", [
    ("read in flight", lambda x: (x.lds("", 100, 4), x.mfma("v[104:107]", "v[100:103]", "v[108:111]", "0"))),
    ("two reads in flight", lambda x: (x.lds("", 100, 4), x.lds("", 102, 4))),
    ("another read", lambda x: (x.lds("", 100, 4, 1), x.lds("", 104, 4, 2), x.wait({100, 104}), x.mfma("v[112:115]", "v[100:103]", "v[104:107]", "0", [("v[104:107]", 3)]))),
    ("too soon behind the MFMA", lambda x: (x.mfma("v[100:103]", "v[104:107]", "v[108:111]", "0"), x.valu("v_mul_f32", "v1", "v100", "v2"))),
    ("MFMA too soon", lambda x: (x.valu("v_mul_f32", "v100", "v1", "v2"), x.mfma("v[104:107]", "v[100:103]", "v[108:111]", "0"))),
    ("transcendental", lambda x: (x.valu("v_exp_f32", "v100", "v1", trans=True), x.valu("v_mul_f32", "v1", "v100", "v2"))),
])
def test_attention_loops_refuse_what_the_hardware_would_not_wait_for(loops, fault, code):
    with pytest.raises(AssertionError, match=fault):
        code(loops.Stream("bf16"))
    x = loops.Stream("bf16")              # waited for, the reads that may be in flight are the younger ones
    x.lds("", 100, 4), x.lds("", 104, 4), x.wait({100})
    assert x.lines[-1] == "s_waitcnt lgkmcnt(1)" and x.reads == [set(range(104, 108))]


def run_stages(lines, stage_bytes, shared, took, rounds=3):
    """Runs a loop's text, following the branches whose label `took` names, and checks the stages of LDS: a copy goes to a stage whose reads have
    all been waited for, and, where wavefronts share a stage, only past a barrier behind that; a read goes to a stage whose copies
    have been waited for, and past a barrier behind that.  The first round only fills the books.  Returns the copies seen."""
    at = {l[:-1]: i for i, l in enumerate(lines) if l.endswith(":")}
    pc, back, seen, copies = at["LLOOP_%="], [], -1, 0
    reads, copying = [], []                       # in flight, oldest first: stages (stores as None)
    unread, landed, ready = set(), set(), set()   # read and not yet known to everyone; landed; landed and known to everyone
    m0 = None
    while True:
        l = lines[pc]
        pc += 1
        if l == "LLOOP_%=:":
            seen += 1
            if seen == rounds:
                return copies
        if l.endswith(":"):
            continue
        op, _, rest = l.partition(" ")
        label = rest.split()[-1] if rest else ""
        if op == "s_branch" or (op.startswith("s_cbranch") and (label in ("LLOOP_%=", "LREST0_%=") or took(label, op))):
            pc = at[label]
            if label == "LREST0_%=":              # the rounds of a wavefront past its rows
                seen += 1
                if seen == rounds:
                    return copies
        elif op == "s_call_b64":
            back.append(pc)
            pc = at[label]
        elif op == "s_setpc_b64":
            pc = back.pop()
        elif op == "s_waitcnt":
            for kind, n in re.findall(r"(vmcnt|lgkmcnt)\((\d+)\)", rest):
                queue = copying if kind == "vmcnt" else reads
                done, queue[:] = queue[:max(0, len(queue) - int(n))], queue[max(0, len(queue) - int(n)):]
                if kind == "vmcnt":
                    landed |= {s for s in done if s is not None and s not in queue}
                if not shared:
                    ready = set(landed)
        elif op == "s_barrier":
            ready, unread = set(landed), set(reads)
        elif op == "s_add_u32" and rest.startswith("m0, "):
            m0 = int(rest.split(", ")[2]) // stage_bytes
        elif op.startswith("buffer_load"):
            if seen > 0:
                assert m0 not in reads and (not shared or m0 not in unread), ("copied over while it is read", m0, lines[pc - 4:pc])
                copies += 1
            copying.append(m0)
            landed.discard(m0), ready.discard(m0)
        elif op.startswith("global_store"):
            copying.append(None)
        elif op.startswith("ds_read") and "%[rk" in rest and not shared:
            reads.append(None)                    # the K tile, which stays
        elif op.startswith("ds_read"):
            stage = int((re.findall(r"offset:(\d+)", rest) or ["0"])[0]) // stage_bytes
            if seen > 0:
                assert stage in ready, ("read before it has landed", stage, lines[pc - 4:pc])
            reads.append(stage)
            if shared:
                unread.add(stage)


def _loop(loops, kind, form):
    x = {"fwd": loops.FWD, "dq": loops.DQ, "dkv": loops.DKV}[kind]("bf16", form)
    return x.text(), x.SLOTB if kind == "dkv" else x.STAGEB


PATHS = {
    "plain": lambda label, op: False,
    "masked": lambda label, op: re.match(r"LMASK", label) is not None,
    "late": lambda label, op: re.match(r"L(MASK|LATE)", label) is not None and op != "s_cbranch_scc0",
    "idle": lambda label, op: re.match(r"L(MASK|LATE|IDLE)", label) is not None and op != "s_cbranch_scc0",
}


@pytest.mark.parametrize("kind,form", [("fwd", 4), ("fwd", 8), ("dq", 4), ("dq", 8), ("dkv", False), ("dkv", True)])
@pytest.mark.parametrize("path", PATHS)
def test_attention_loops_copy_to_stages_that_nobody_reads(loops, kind, form, path):
    text, stage = _loop(loops, kind, form)
    assert run_stages(text, stage, kind != "dkv", PATHS[path]) >= 16


@pytest.mark.parametrize("kind,form,was,becomes,what", [
    ("fwd", 4, "s_waitcnt vmcnt(4)", "s_waitcnt vmcnt(8)", "landed"), ("dq", 8, "s_waitcnt vmcnt(16)", "s_waitcnt vmcnt(24)", "landed"),
    ("dkv", True, "s_waitcnt vmcnt(8)", "s_waitcnt vmcnt(12)", "landed"), ("fwd", 4, "s_barrier", "s_nop 0", "read"),
    ("dq", 4, "s_barrier", "s_nop 0", "read")])
def test_attention_loops_with_a_wait_less_are_found(loops, kind, form, was, becomes, what):
    text, stage = _loop(loops, kind, form)
    assert was in text
    with pytest.raises(AssertionError, match=what):
        run_stages([becomes if l == was else l for l in text], stage, kind != "dkv", PATHS["plain"])


def test_attention_loops_name_what_they_change(loops):
    """Scalar condition and m0 as well: a value of the compiler's must not live across a loop in them."""
    names = [l for l in loops.generate().split("\n") if "_CLOBBERS" in l]
    assert len(names) == 3 and all(all('"%s"' % r in l for r in ("vcc", "scc", "m0", "memory")) for l in names)
