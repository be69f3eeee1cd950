"""The C-ABI library loads and exports every symbol the header declares (no GPU needed)."""
import ctypes
import os
import re

import pytest

from dhellam_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "dhellam_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(dh_[a-z0-9_]+)\s*\(", text)))


def _ensure_lib():
    if not _lib.LIB_PATH.exists():
        from dhellam_amd.build import build
        build()


def test_header_and_ctypes_table_agree():
    assert _declared_symbols() == sorted(_lib.SIGNATURES), "include/dhellam_hip.h and _lib.SIGNATURES list different symbols"


def test_library_exports_every_declared_symbol():
    _ensure_lib()
    lib = ctypes.CDLL(str(_lib.LIB_PATH))
    for name in _declared_symbols():
        assert hasattr(lib, name), f"{name} is declared in the header but missing from the library"


def test_argument_counts_match_header():
    text = open(os.path.join(ROOT, "include", "dhellam_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    for name, (_, args) in _lib.SIGNATURES.items():
        m = re.search(r"\b%s\s*\(([^;]*?)\)\s*;" % name, text, flags=re.S)
        assert m, name
        params = m.group(1).strip()
        n = 0 if params in ("", "void") else len([p for p in params.split(",") if p.strip()])
        assert n == len(args), f"{name}: header has {n} parameters, ctypes table has {len(args)}"


def test_version_and_error_string_without_gpu():
    _ensure_lib()
    lib = _lib.load()
    assert lib.dh_version() >= 100
    # argument validation happens on the host, before any HIP call: usable without a GPU
    rc = lib.dh_norm_fwd(None, None, None, None, None, None, 4, 0, 1e-5, 0, 0, None)
    assert rc == -1
    msg = lib.dh_last_error().decode()
    assert "norm.hip" in msg and "norm_fwd" in msg and "bad shape" in msg
    rc = lib.dh_attn_fwd(None, None, None, None, None, None, None, 1, 8, 8, 5, 2, 64, 0, 0, 0, 0, 1.0, 1, 1, None)
    assert rc == -1 and "multiple" in lib.dh_last_error().decode()
    rc = lib.dh_moe_route_topk(None, None, None, 10, 100, 2, None)
    assert rc == -1 and "experts" in lib.dh_last_error().decode()


@pytest.mark.parametrize("batch,max_q,total_q,hq,causal,hand", [
    (4, 2048, 8192, 8, 1, True), (4, 2048, 8192 - 1300, 8, 1, False),        # one round of workgroups; 84 % of one
    (7, 3324, 8192, 32, 1, True), (5, 1423, 2118, 32, 1, False),             # several lengths: four rounds of work; one of short rows
    (1, 4352, 4352, 32, 1, False), (32, 300, 9600, 16, 1, False),            # two rounds and an eighth; short rows
    (1, 4096, 4096, 8, 1, True), (4, 1024, 4096, 8, 1, False),               # 64-row tiles: long and short rows
    (1, 384, 384, 16, 0, True), (1, 384, 384, 15, 0, False),                 # not causal: 96 and 90 workgroups
    (0, 0, 0, 8, 1, False), (3, 0, 0, 8, 1, False), (2, 4096, 0, 64, 1, False), (1, 4096, 1 << 40, 8, 1, True),
])
def test_attention_route(batch, max_q, total_q, hq, causal, hand):
    """Both sides of the lines between the two families of head-dim-128 kernels, and sizes at which nothing is left to divide."""
    _ensure_lib()
    lib = _lib.load()
    assert bool(lib.dh_attn_fwd_path(batch, max_q, total_q, hq, 128, causal) & 1) == hand
    assert lib.dh_attn_fwd_path(batch, max_q, total_q, hq, 96, causal) & 1 == 0
    assert lib.dh_attn_bwd_path(batch, max_q, max_q, total_q, total_q, hq, hq, 96, causal, 1 << 40) & 7 == 0


@pytest.mark.parametrize("batch,max_q,max_k,total_q,hq,causal,fwd,dq", [
    (1, 4096, 4096, 4096, 32, 1, 256, 256), (1, 2048, 2048, 2048, 32, 1, 0, 128), (1, 2689, 2689, 2689, 20, 1, 128, 0),
    (1, 700, 2000, 700, 44, 0, 128, 128), (1, 700, 700, 700, 44, 0, 0, 256),                 # the forward by the number of keys
    (1, 1284, 1284, 1284, 12, 0, 0, 0), (1, 1363, 1363, 1363, 12, 0, 128, 0), (6, 512, 512, 3072, 64, 1, 0, 256),          # the forward's rounds
    (1, 3003, 3003, 3003, 64, 1, 128, 128), (5, 4799, 4799, 23995, 4, 0, 128, 128), (32, 605, 605, 12640, 16, 1, 0, 256),
    (8, 812, 812, 4464, 64, 1, 256, 256),
    (1, 600, 333, 600, 32, 0, 128, 0), (0, 0, 0, 0, 8, 1, 0, 0), (1, 4096, 0, 4096, 32, 0, 256, 256),
    (5, 628, 628, 3140, 32, 1, 0, 128), (16, 512, 512, 8192, 16, 1, 256, 256), (8, 1024, 1024, 8192, 32, 1, 256, 256),     # dQ: rounds of work
    (8, 96, 96, 768, 32, 0, 0, 0), (12, 140, 140, 1680, 16, 0, 0, 256), (1, 2048, 333, 2048, 16, 0, 0, 128), (1, 2048, 20, 2048, 16, 0, 0, 0)])
def test_attention_tiles_on_one_wavefront_a_simd(batch, max_q, max_k, total_q, hq, causal, fwd, dq):
    """Head dim 128 without room for dS: query rows of a tile, forward and dQ, on both sides of the lines."""
    _ensure_lib()
    lib = _lib.load()
    assert lib.dh_attn_fwd_rows(batch, max_q, max_k, total_q, hq, 128, causal) == fwd
    assert lib.dh_attn_bwd_dq_rows(batch, max_q, max_k, total_q, total_q, hq, hq, 128, causal, 0) == dq
    assert lib.dh_attn_fwd_rows(batch, max_q, max_k, total_q, hq, 96, causal) == 0
    if max_q == max_k:
        assert bool(lib.dh_attn_fwd_path(batch, max_q, total_q, hq, 128, causal) & 4) == (fwd > 0)


@pytest.mark.parametrize("lens,hq,hk,one,path", [
    ([1000] + [1] * 7, 8, 8, 1, 0), ([1500] + [20] * 15, 4, 4, 1, 0), ([386, 382] + [1] * 14, 12, 4, 1, 0),
    ([599] + [1] * 47, 4, 4, 0, 9), ([599] + [1] * 23, 4, 4, 1, 0)])
def test_attention_backward_of_one_long_sequence_among_many_short_ones(lens, hq, hk, one, path):
    """The one launch, or the hand-ordered dK/dV (1; 8: with 128-row dQ tiles): not the other kernels in two launches."""
    _ensure_lib()
    lib = _lib.load()
    sizes = len(lens), max(lens), max(lens), sum(lens), sum(lens), hq, hk, 128, 1
    assert lib.dh_attn_bwd_one_launch(*sizes) == one
    assert lib.dh_attn_bwd_path(*sizes, 1 << 40) == path


@pytest.mark.parametrize("q,k,one", [(12, 7147, 0), (363, 1427, 0), (44, 601, 0), (44, 600, 1), (600, 900, 1), (600, 901, 0), (3000, 20, 1)])
def test_attention_backward_of_few_rows_and_many_keys(q, k, one):
    """At head dim 128, not causal: dQ of a few rows over many keys is not left to the few workgroups of the one launch."""
    _ensure_lib()
    assert _lib.load().dh_attn_bwd_one_launch(1, q, k, q, k, 1, 1, 128, 0) == one


def test_product_does_not_import_the_oracle():
    """Nothing under dhellam_amd/ may import, read or run the oracle (it is the checker)."""
    for dirpath, _, files in list(os.walk(os.path.join(ROOT, "dhellam_amd"))) + list(os.walk(os.path.join(ROOT, "dhellam"))):
        for f in files:
            if f.endswith((".py", ".hip", ".h")):
                src = open(os.path.join(dirpath, f)).read()
                assert not re.search(r"^\s*(from|import)\s+oracle\b", src, flags=re.M), f"{f} imports the oracle"
