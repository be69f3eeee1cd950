"""Build-time checks that need no GPU."""
import shutil

import pytest


@pytest.mark.skipif(shutil.which("hipcc") is None and not __import__("os").path.exists("/opt/rocm/bin/hipcc"),
                    reason="needs hipcc")
def test_grouped_gemm_loads_are_left_alone_until_used():
    """The chip-filling grouped GEMM copies its operands to LDS from assembly and orders reads, waits, copies and barriers
    by hand: the compiled loop has to keep that order, without spills, in all of the ten instantiations (NT / NN with and
    without the split last round, TN; bf16 and fp16).  ``check_grouped_gemm_loops`` compiles the source to assembly and
    verifies that; a violation raises."""
    from dhellam_amd.build import check_grouped_gemm_loops
    assert check_grouped_gemm_loops() == 10


def test_weight_gradients_of_very_long_rows_stay_with_the_library():
    """The grouped kernel's tiles address rows of fewer than 2^22 elements."""
    from dhellam_amd import _host
    edge = (1 << 22) - 8
    assert _host.wgrad_grouped(16, edge, 256) and _host.wgrad_grouped(16, 256, edge)
    assert not _host.wgrad_grouped(16, edge + 8, 256) and not _host.wgrad_grouped(16, 256, edge + 8)
    assert not _host.wgrad_grouped(16, 5000000, 256)
