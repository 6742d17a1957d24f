"""Build libstrict_topk_hip.so for gfx950 with hipcc (in-tree).

Usage: python strict-topk-overlap_amd/build_lib.py [--jobs N]

Objects go to strict-topk-overlap_amd/_build/, the shared library and the native
host module next to the Python package (strict_topk/libstrict_topk_hip.so,
strict_topk/_host.<python tag>.so), so they travel with the source tree.
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import re
import shutil
import subprocess
import sys
import sysconfig
import tempfile
from pathlib import Path

ROOT = Path(__file__).resolve().parent
CSRC = ROOT / "csrc"
OUT = ROOT / "strict_topk" / "libstrict_topk_hip.so"
HOST = ROOT / "strict_topk" / ("_host" + sysconfig.get_config_var("EXT_SUFFIX"))
BUILD = ROOT / "_build"
ARCH = "gfx950"
SOURCES = ["api.cpp", "states.hip", "select.hip", "repair.hip", "signed.hip", "hier.hip", "sstep.hip",
           "bounds.hip", "indexer.hip", "paged.hip", "step.hip", "tail_dense.hip", "front_pg.hip",
           "tail_pg.hip", "stail_pg.hip", "cache.hip", "srepair.hip", "srepair_compact.hip", "compact.hip",
           "hier_mfma.hip", "step1.hip", "repair_fast.hip", "step_small.hip"]

FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    "-Wall", "-Wno-unused-function", "-Wno-unknown-warning-option",
    # packed FP32 ops stay disabled for every HIP translation unit
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def hipcc():
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found")


def _up_to_date(src: str, obj: Path) -> bool:
    """STK_INCREMENTAL=1 (development only): an object newer than its source
    and every header is kept."""
    if not os.environ.get("STK_INCREMENTAL") or not obj.exists():
        return False
    deps = [CSRC / src, *CSRC.glob("*.hpp"), ROOT.parent / "include" / "strict_topk.h"]
    return obj.stat().st_mtime > max(d.stat().st_mtime for d in deps)


def _compile(src: str) -> Path:
    obj = BUILD / (Path(src).stem + ".o")
    if _up_to_date(src, obj):
        return obj
    lang = ["-x", "hip"] if src.endswith(".hip") else []
    with tempfile.TemporaryDirectory(dir=BUILD) as tmp:
        out = Path(tmp) / obj.name
        keep = ["-save-temps=obj"] if lang else []
        cmd = [hipcc(), *FLAGS, *keep, *lang, "-c", str(CSRC / src), "-o", str(out)]
        res = subprocess.run(cmd, capture_output=True, text=True)
        noise = "packed-fp32-ops"
        err = "\n".join(l for l in res.stderr.splitlines() if noise not in l)
        if res.returncode != 0:
            raise RuntimeError(f"hipcc failed for {src}:\n{err}")
        for asm in Path(tmp).glob(f"*-{ARCH}.s"):
            bad = misplaced_copies(asm.read_text().splitlines())
            if bad:
                raise RuntimeError(f"{src}: register copies ahead of an exec restore (wrong "
                                   "values in lanes that skip the branch); change the kernel's "
                                   "register layout:\n" + "\n".join(bad))
        os.replace(out, obj)
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def misplaced_copies(lines) -> list[str]:
    """Places in gfx950 assembly where the compiler copies, spills or reloads a
    vector register at the head of a join block, ahead of the instruction that
    gives the lanes that skipped the branch their exec bits back: in those lanes
    the copy is not made.  (Seen in a kernel that fills the register file: the
    allocator put its copy before scalar copies that it had put before the
    restore.  The sums of a wave whose rows were all skipped went to a wrong LDS
    address.)"""
    joins = {m[1] for l in lines if (m := re.match(r"\s+s_cbranch_execz (\S+)", l))}
    block = re.compile(r"(\.LBB\d+_\d+):|; %bb\.\d+:")
    copy = re.compile(r"(v_mov_b(32|64)_e32 v\S+ v|v_accvgpr_|scratch_(load|store)_)")
    bad, pending, watch, fn, last = [], [], False, "", ""
    for i, line in enumerate(lines, 1):
        if m := block.match(line):
            # a block without a label joins what it follows, unless a branch to
            # the join just skipped it: then it is the branch's body
            watch = m[1] in joins if m[1] else not last.startswith("s_cbranch_exec")
            pending = []
            continue
        text = line.split(";")[0].strip()
        if m := re.match(r"(_Z\w+):", text):
            fn, watch = m[1], False
        if not text or text.startswith("."):
            continue
        last = text
        if not watch:
            continue
        if text.startswith("s_or_b64 exec, exec, "):
            bad += [f"{fn} line {n}: {t}" for n, t in pending]
            watch = False
        elif re.match(r"s_\w+ exec,|s_\w+saveexec|s_c?branch", text):
            watch = False
        elif copy.match(text):
            pending.append((i, text))
    return bad


def build_host() -> Path:
    """The native host path (csrc/host.cpp), a Python extension module over
    torch's C++ tensors; no device code."""
    import torch
    root = Path(torch.__file__).resolve().parent
    tmp = HOST.with_suffix(".so.tmp")
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall",
           "-Wno-sign-compare", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           f'-DSTK_TORCH_VERSION="{torch.__version__}"',
           f"-isystem{root / 'include'}",
           f"-isystem{root / 'include' / 'torch' / 'csrc' / 'api' / 'include'}",
           "-isystem/opt/rocm/include", f"-isystem{sysconfig.get_path('include')}",
           str(CSRC / "host.cpp"), "-o", str(tmp), f"-L{root / 'lib'}", "-ltorch_python",
           "-ltorch_cpu", "-ltorch", "-lc10", "-lc10_hip"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"host module failed:\n{res.stderr}")
    os.replace(tmp, HOST)
    # a module without the tag would be loaded by any Python
    (HOST.parent / "_host.so").unlink(missing_ok=True)
    return HOST


def build(jobs: int | None = None) -> Path:
    BUILD.mkdir(exist_ok=True)
    jobs = jobs or min(len(SOURCES), os.cpu_count() or 4)
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        host = ex.submit(build_host)
        objs = list(ex.map(_compile, SOURCES))
        host.result()
    tmp = OUT.with_suffix(".so.tmp")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp),
           *map(str, objs)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    os.replace(tmp, OUT)
    return OUT


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=None)
    args = ap.parse_args()
    print(build(args.jobs))
