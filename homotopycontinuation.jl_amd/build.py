"""Builds libhcgpu.so in-tree (homotopycontinuation.jl_amd/_build/).

1. Embeds the device headers (csrc/device/*.h and include/hcgpu_types.h) as C++ raw strings
   into csrc/_gen/device_headers.inc; hipRTC compiles every generated program
   against them at hcg_program_create time.
2. Compiles the host runtime, the code generator and the MLP training kernels with
   hipcc for gfx950.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
REPO = PKG.parent
CSRC = PKG / "csrc"
OUT = PKG / "_build"
HEADERS = [
    ("hcg_arith.h", CSRC / "device" / "hcg_arith.h"),
    ("hcg_tracker.h", CSRC / "device" / "hcg_tracker.h"),
    ("hcg_tracker_body.h", CSRC / "device" / "hcg_tracker_body.h"),
    ("hcg_learned.h", CSRC / "device" / "hcg_learned.h"),
    ("hcg_mlp_infer.h", CSRC / "device" / "hcg_mlp_infer.h"),
    ("hcg_kargs.h", CSRC / "device" / "hcg_kargs.h"),
    ("hcg_sched.h", CSRC / "device" / "hcg_sched.h"),
    ("hcg_interval.h", CSRC / "device" / "hcg_interval.h"),
    ("hcg_certify.h", CSRC / "device" / "hcg_certify.h"),
    ("hcg_cert_kargs.h", CSRC / "device" / "hcg_cert_kargs.h"),
    ("hcgpu_types.h", REPO / "include" / "hcgpu_types.h"),
]
DELIM = "HCGRAWSRC"


def write_header_inc():
    gen = CSRC / "_gen"
    gen.mkdir(exist_ok=True)
    names, srcs = [], []
    for name, path in HEADERS:
        text = path.read_text()
        if f"){DELIM}\"" in text:
            raise RuntimeError(f"raw-string delimiter occurs in {path}")
        names.append(f'"{name}"')
        # split into chunks to stay below compiler string-literal limits
        chunks = [text[i:i + 12000] for i in range(0, len(text), 12000)] or [""]
        srcs.append("\n".join(f'R"{DELIM}({c}){DELIM}"' for c in chunks))
    body = "// generated by build.py: device headers compiled by hipRTC\n"
    body += "static const char* k_hdr_names[] = {" + ", ".join(names) + "};\n"
    body += "static const char* k_hdr_srcs[] = {\n" + ",\n".join(srcs) + "\n};\n"
    target = gen / "device_headers.inc"
    if not target.exists() or target.read_text() != body:
        target.write_text(body)


def hipcc():
    for c in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if c and os.path.exists(c):
            return c
    raise RuntimeError("hipcc not found")


SOURCES = ["hcgpu.cpp", "codegen.cpp", "mlp.hip", "noalloc.hip", "group_sched.cpp", "group.cpp", "group_kernel.hip",
           "group_kernel32.hip", "group_kernel32_wide.hip"]
# -ffp-contract=off: FMAs only where the code writes fma(), the arithmetic contract the oracle and
# the hipRTC-compiled kernels share (results equal the oracle's bit for bit)
FLAGS = ["-O3", "-fPIC", "-std=c++17", "--offload-arch=gfx950", "-ffp-contract=off", "-Xclang", "-target-feature",
         "-Xclang", "-packed-fp32-ops", "-Wno-unused-result", "-Wno-unused-command-line-argument"]


def _newest_header() -> float:
    paths = list((CSRC / "device").glob("*.h")) + list(CSRC.glob("*.h")) + list((REPO / "include").glob("*.h"))
    paths.append(CSRC / "_gen" / "device_headers.inc")
    return max(p.stat().st_mtime for p in paths if p.exists())


def build(verbose: bool = False, incremental: bool = False) -> Path:
    """Compile every source of libhcgpu.so (in parallel, one object each) and link it.
    incremental=True keeps objects newer than their source and every header."""
    from concurrent.futures import ThreadPoolExecutor
    write_header_inc()
    OUT.mkdir(exist_ok=True)
    objdir = OUT / "obj"
    objdir.mkdir(exist_ok=True)
    inc = [f"-I{REPO / 'include'}", f"-I{CSRC}"]
    hdr = _newest_header()

    def compile_one(src: str) -> Path:
        obj = objdir / (src.replace(".", "_") + ".o")
        if incremental and obj.exists() and obj.stat().st_mtime > max(hdr, (CSRC / src).stat().st_mtime):
            return obj
        cmd = [hipcc(), *FLAGS, *inc, "-c", str(CSRC / src), "-o", str(obj) + ".tmp"]
        if verbose:
            print(" ".join(cmd), flush=True)
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            sys.stderr.write(r.stdout + r.stderr)
            raise RuntimeError(f"hipcc failed on {src}")
        os.replace(str(obj) + ".tmp", obj)
        return obj

    # the lane-group kernels take longest: start them first
    order = sorted(SOURCES, key=lambda s: 0 if s.startswith("group_kernel") else 1)
    with ThreadPoolExecutor(max_workers=min(len(order), os.cpu_count() or 1)) as pool:
        objs = list(pool.map(compile_one, order))
    lib = OUT / "libhcgpu.so"
    tmp = OUT / "libhcgpu.so.tmp"
    cmd = [hipcc(), *FLAGS, "-shared", *[str(o) for o in objs], "-lhiprtc", "-o", str(tmp)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("hipcc failed linking libhcgpu.so")
    os.replace(tmp, lib)
    return lib


if __name__ == "__main__":
    print(build(verbose=True, incremental="--incremental" in sys.argv))
