"""Builds the gfx950 operator library (``libdhellam_hip.so``) with hipcc.

The library is plain HIP behind a C ABI (``include/dhellam_hip.h``): no torch
headers, so a cross-compile needs only ROCm.  Objects go to ``build/`` and the
shared object to ``dhellam_amd/lib/`` (in-tree, so it is found next to the
package without installation).

Run as ``python -m dhellam_amd.build``.
"""
from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
LIB_DIR = PKG / "lib"
LIB_PATH = LIB_DIR / "libdhellam_hip.so"
OBJ_DIR = ROOT / "build" / "obj"
GEN_DIR = ROOT / "build" / "gen"          # sources that are written by programs: attn_loops.inc

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

# -packed-fp32-ops is switched off: the compiler would otherwise form packed
# fp32 VALU instructions from scalar float code.
CXXFLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-gpu-rdc",
    "-Wall",
    "-Wno-unused-function",
    "-Wno-unknown-pragmas",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    f"-I{ROOT / 'include'}",
    f"-I{GEN_DIR}",
]


def sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip"))


def generate_sources() -> None:
    """Writes ``attn_loops.inc``: the main loops of the attention kernels with one wavefront on a SIMD (``csrc/attn_loops.py``)."""
    GEN_DIR.mkdir(parents=True, exist_ok=True)
    subprocess.run([sys.executable, str(CSRC / "attn_loops.py"), str(GEN_DIR / "attn_loops.inc")], check=True)


def _compile(src: Path, verbose: bool) -> Path:
    obj = OBJ_DIR / (src.stem + ".o")
    cmd = [HIPCC, *CXXFLAGS, "-c", str(src), "-o", str(obj)]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    # hipcc's host pass warns that it does not know the packed-fp32 feature; drop that line.
    err = "\n".join(l for l in res.stderr.splitlines() if "packed-fp32-ops" not in l)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{err}")
    if err.strip() and verbose:
        print(err, file=sys.stderr)
    return obj


def build(verbose: bool = False, jobs: int | None = None) -> Path:
    """Compile every ``csrc/*.hip`` for gfx950 and link the shared library."""
    OBJ_DIR.mkdir(parents=True, exist_ok=True)
    LIB_DIR.mkdir(parents=True, exist_ok=True)
    generate_sources()
    srcs = sources()
    if not srcs:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    jobs = jobs or min(8, len(srcs), os.cpu_count() or 1)
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(lambda s: _compile(s, verbose), srcs))
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-fno-gpu-rdc",
           *map(str, objs), "-lhipblaslt", "-o", str(tmp)]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    os.replace(tmp, LIB_PATH)
    return LIB_PATH


def grouped_gemm_assembly() -> list:
    """The instantiations of ``grouped_gemm_w8_kernel`` as device assembly of ``grouped_gemm.hip``, a list of lines each."""
    import re
    import tempfile
    with tempfile.TemporaryDirectory() as td:
        out = Path(td) / "gg.s"
        cmd = [HIPCC, *[f for f in CXXFLAGS if f != "-fPIC"], "--cuda-device-only", "-S", str(CSRC / "grouped_gemm.hip"), "-o", str(out)]
        res = subprocess.run(cmd, capture_output=True, text=True)
        if res.returncode != 0:
            raise RuntimeError("hipcc -S failed for grouped_gemm.hip:\n" + res.stderr)
        lines = out.read_text().split("\n")
    starts = [i for i, l in enumerate(lines) if re.match(r"^_ZN2dh22grouped_gemm_w8_kernel\w+:", l)]
    if not starts:
        raise RuntimeError("no grouped_gemm_w8_kernel instantiation found in the assembly")
    # (a kernel may hold several s_endpgm)
    return [lines[a:next(i for i in range(a, len(lines)) if lines[i].startswith(".Lfunc_end"))] for a in starts]


def check_grouped_gemm_loops(verbose: bool = False) -> int:
    """The chip-filling grouped GEMM kernel (``grouped_gemm_w8_kernel``) copies its operands to LDS from assembly, which
    the compiler does not count: that no copy overtakes a fragment read and no read a copy rests on the order of reads,
    waits, copies and barriers that the source lays down.  This holds the generated code of every instantiation to it
    (``check_grouped_gemm_order``).  Returns the number of instantiations checked; raises on a violation."""
    kernels = grouped_gemm_assembly()
    for fn in kernels:
        body = check_grouped_gemm_order(fn)
        if verbose:
            print(f"checked {fn[0].split(':')[0]}: {body} lines", flush=True)
    return len(kernels)


def check_grouped_gemm_order(fn: list) -> int:
    """One instantiation of ``grouped_gemm_w8_kernel`` as assembly: the copies of the first two slices, published by the
    counted wait and a barrier before anything is read, and one more barrier for half of the wavefronts; the main loop (the
    innermost loop with 128 MFMAs: two slices) and, behind it, the last slice of an odd number.  In the slices, cut at their
    barriers, clusters of 16 MFMAs have to alternate with clusters of none, copies may stand in the latter only, each of these
    has to begin by waiting for the wavefront's earlier LDS reads, and where copies are published the wait for them is the one
    the source counts.  Behind the last slice everything has landed, past a barrier, before LDS is used again.  No scratch
    accesses, no copies of accumulators, and no register moves among MFMAs.  Returns the lines of the loop."""
    import re
    name = fn[0].split(":")[0]
    code = [l.split(";")[0].strip() for l in fn]
    labels = {m.group(1): i for i, l in enumerate(code) if (m := re.match(r"^(\.LBB\d+_\d+):", l))}
    mfmas = lambda part: sum("v_mfma" in x for x in part)
    barriers = lambda part: [i for i, x in enumerate(part) if x.startswith("s_barrier")]
    copies = lambda part: [i for i, x in enumerate(part) if x.startswith("buffer_load")]

    def need(ok, what):
        if not ok:
            raise RuntimeError(f"{name}: {what}")

    loops = []
    for i, l in enumerate(code):
        m = re.match(r"s_c?branch\w* (\.LBB\d+_\d+)", l)
        if m and m.group(1) in labels and labels[m.group(1)] < i and mfmas(code[labels[m.group(1)] + 1:i]) == 128:
            loops.append((labels[m.group(1)] + 1, i))
    need(loops, "no main loop with 128 MFMAs found (the kernel's structure changed: update check_grouped_gemm_order)")
    lo, hi = min(loops, key=lambda x: x[1] - x[0])
    plain = lambda part: [x for x in part if x and not x.endswith(":")]
    first, body, rest = plain(code[:lo]), plain(code[lo:hi]), plain(code[hi:])
    need(mfmas(first) == 0 and mfmas(rest) == 64, f"{mfmas(first)} and {mfmas(rest)} MFMAs before and behind the main loop, expected 0 and 64")

    def check_slices(clusters, where):
        total = 0
        for n, cl in enumerate(clusters):
            dma = copies(cl)
            need(mfmas(cl) == (16 if n % 2 else 0), f"{where}: cluster {n} holds {mfmas(cl)} MFMAs")
            need(not any("scratch_" in x or "v_accvgpr" in x for x in cl), f"{where}: scratch or accumulator copies in cluster {n}")
            total += len(dma)
            if n % 2:
                need(not dma, f"{where}: a copy among the MFMAs of cluster {n}")
                need(not any(x.startswith("v_mov_b") for x in cl), f"{where}: a register move among the MFMAs of cluster {n}")
                continue
            waits = [i for i, x in enumerate(cl) if x == "s_waitcnt lgkmcnt(0)"]
            reads = [i for i, x in enumerate(cl) if x.startswith("ds_read")]
            need(waits and not (reads and reads[0] < waits[0]) and not (dma and dma[0] < waits[0]),
                 f"{where}: cluster {n} does not begin with the wait for the earlier reads")
            need(all(cl[i].endswith("lds") for i in dma), f"{where}: a load to registers in cluster {n}")
            need(not dma or "s_waitcnt vmcnt(8)" in cl[dma[-1]:], f"{where}: cluster {n} publishes copies without the counted wait")
        need(total == len(clusters), f"{where}: {total} copies, expected {len(clusters)}")

    def cut(part):
        at = [-1] + barriers(part)
        return [part[x + 1:y] for x, y in zip(at, at[1:])], part[at[-1] + 1:]

    # the first two slices
    dma = copies(first)
    need(len(dma) == 16 and all(first[i].endswith("lds") for i in dma), f"{len(dma)} loads before the main loop, expected 16 copies")
    need("s_waitcnt vmcnt(0)" in first[:dma[0]], "the stores before the first copies are not waited for")
    behind = first[dma[-1] + 1:]
    bars = barriers(behind)
    need(len(bars) == 2, f"{len(bars)} barriers between the first copies and the main loop, expected 2")
    need("s_waitcnt vmcnt(8)" in behind[:bars[0]], "the first slice is published without the counted wait")
    reads = [i for i, x in enumerate(first) if x.startswith("ds_read")]
    need(reads and reads[0] > dma[-1] + 1 + bars[1], "a fragment is read before the first slice is published")
    # the loop
    clusters, head = cut(body)
    need(len(clusters) == 16, f"{len(clusters)} barriers in the main loop, expected 16")
    clusters[0] = head + clusters[0]                     # what follows the last barrier runs into the loop's head
    check_slices(clusters, "main loop")
    # the last slice of an odd number
    at = barriers(rest)
    need(len(at) >= 10, f"{len(at)} barriers behind the main loop, expected 10 and more")
    clusters, _ = cut(rest[:at[7] + 1])
    waits = [i for i, x in enumerate(clusters[0]) if x == "s_waitcnt lgkmcnt(0)"]    # (the blocks that the branches over it lead to)
    need(waits and not any(x.startswith("ds_read") for x in clusters[0][:waits[-1]]), "last slice: a read before the wait for the earlier ones")
    clusters[0] = clusters[0][waits[-1]:]
    check_slices(clusters, "last slice")
    # and what follows: the other half's barrier, the last copies, a barrier, and only then LDS again
    behind = rest[at[7] + 1:]
    used = next((i for i, x in enumerate(behind) if x.startswith(("ds_", "global_store", "buffer_load"))), len(behind))
    landed = next((i for i, x in enumerate(behind) if re.match(r"s_waitcnt vmcnt\(0\)", x)), len(behind))
    need(landed < used and any(landed < i < used for i in barriers(behind)), "LDS is used again before the last copies have landed")
    return len(body)


EXT_PKG = ROOT / "dhellam"
EXT_SUFFIX = sysconfig.get_config_var("EXT_SUFFIX")
PY_INCLUDE = sysconfig.get_paths()["include"]


def torch_extension_path() -> Path:
    return EXT_PKG / ("_Clib" + EXT_SUFFIX)


def host_extension_path() -> Path:
    return PKG / ("_host" + EXT_SUFFIX)


def _build_extension(src: Path, out: Path, rpath: str, verbose: bool) -> Path:
    """Host code only: the host compiler with torch's headers, linked against ``libdhellam_hip.so`` (found at run
    time relative to the extension)."""
    import torch
    from torch.utils import cpp_extension as E
    if not LIB_PATH.exists():
        raise RuntimeError(f"{LIB_PATH} must be built first")
    rocm = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))
    name = out.name.split(".")[0]
    tmp = out.with_suffix(".so.tmp")
    torch_lib = E.library_paths()[0]
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Wno-unused-function",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f"-DTORCH_EXTENSION_NAME={name}", "-DTORCH_API_INCLUDE_EXTENSION_H",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           f"-I{ROOT / 'include'}", *[f"-isystem{p}" for p in E.include_paths()], f"-isystem{rocm / 'include'}",
           f"-I{PY_INCLUDE}", str(src), "-o", str(tmp),
           f"-L{torch_lib}", "-lc10", "-lc10_hip", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-ltorch_python", "-lamdhip64",
           f"-L{LIB_DIR}", "-ldhellam_hip", f"-Wl,-rpath,{rpath}", f"-Wl,-rpath,{torch_lib}"]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"building {name} failed:\n{res.stderr}")
    if res.stderr.strip() and verbose:
        print(res.stderr, file=sys.stderr)
    os.replace(tmp, out)
    return out


def build_torch_extension(verbose: bool = False) -> Path:
    """Compiles ``csrc/torchapi.cpp`` into the pybind11 torch extension ``dhellam._Clib`` (the reference builds a
    module of that name from its csrc/torchapi.cpp, setup.py:234-244)."""
    return _build_extension(CSRC / "torchapi.cpp", torch_extension_path(), "$ORIGIN/../dhellam_amd/lib", verbose)


def build_host_extension(verbose: bool = False) -> Path:
    """Compiles ``csrc/hostapi.cpp`` into ``dhellam_amd._host``, the host path of the Python operators."""
    return _build_extension(CSRC / "hostapi.cpp", host_extension_path(), "$ORIGIN/lib", verbose)


def build_extensions(verbose: bool = False) -> list[Path]:
    """Both extensions, side by side."""
    with ThreadPoolExecutor(max_workers=2) as ex:
        return [f.result() for f in [ex.submit(build_host_extension, verbose), ex.submit(build_torch_extension, verbose)]]


if __name__ == "__main__":
    path = build(verbose="-v" in sys.argv)
    print(path)
    print(f"grouped GEMM main loops checked: {check_grouped_gemm_loops(verbose='-v' in sys.argv)}")
    if "--no-ext" not in sys.argv:
        for path in build_extensions(verbose="-v" in sys.argv):
            print(path)
