"""Build recipe of libtsi.so (HIP for gfx950) -- used by __graft_entry__.build().

The library is built in-tree (temporalsetinversion_amd/_build/libtsi.so) so that it
travels with the source tree.  Floating-point rules: no FMA contraction, IEEE division
and square root (hipcc defaults), packed-FP32 instructions disabled.
"""
from __future__ import annotations

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT_DIR = os.path.join(HERE, "_build")
LIB = os.path.join(OUT_DIR, "libtsi.so")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")

SOURCES = ["tsi_kernels.hip", "tsi_trace.hip", "tsi_runtime.hip", "tsi_batch.hip", "tsi_hostmem.hip", "tsi_lower.cpp", "tsi_ir.cpp", "tsi_jit.cpp", "tsi_png.cpp"]
# headers the per-tape kernels are compiled against at run time (embedded in the library)
JIT_HEADERS = ["tsi_interval.h", "tsi_tape.h", "tsi_kernels.h", "tsi_wave.h", "tsi_rules.h", "tsi_eval.h",
               "tsi_batch.h"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("TSI_OFFLOAD_ARCH", "gfx950")

FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unused-variable",
    # the tape interpreter's opcode dispatch is wave-uniform: keep it as scalar branches
    # instead of exec-mask flow blocks
    "-mllvm", "-structurizecfg-skip-uniform-regions=true",
]


def _embed_headers() -> str:
    """Writes _build/tsi_jit_headers.cpp: the JIT headers as C strings."""
    out = os.path.join(OUT_DIR, "tsi_jit_headers.cpp")
    lines = ["// generated by build.py: kernel headers for hiprtc", 'extern "C" {',
             f"extern const int tsi_jit_num_headers = {len(JIT_HEADERS)};",
             "extern const char *const tsi_jit_header_names[] = {" + ", ".join(f'"{h}"' for h in JIT_HEADERS) + "};",
             "extern const char *const tsi_jit_header_texts[] = {"]
    for h in JIT_HEADERS:
        with open(os.path.join(CSRC, h)) as f:
            text = f.read()
        if ")tsi_hdr\"" in text:
            raise RuntimeError(f"{h} contains the raw-string delimiter")
        lines.append('R"tsi_hdr(' + text + ')tsi_hdr",')
    lines += ["};", "}"]
    with open(out, "w") as f:
        f.write("\n".join(lines) + "\n")
    return out


def build(verbose: bool = False) -> str:
    os.makedirs(OUT_DIR, exist_ok=True)
    objs = []
    hdr_src = _embed_headers()
    hdr_obj = os.path.join(OUT_DIR, "tsi_jit_headers.o")
    r = subprocess.run(["g++", "-O1", "-fPIC", "-c", hdr_src, "-o", hdr_obj], capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("embedding the kernel headers failed")
    objs.append(hdr_obj)
    for src in SOURCES:
        obj = os.path.join(OUT_DIR, os.path.splitext(src)[0] + ".o")
        lang = ["-x", "hip"] if src.endswith(".hip") else []
        cmd = [HIPCC, *FLAGS, "-I", INCLUDE, "-I", CSRC, *lang, "-c", os.path.join(CSRC, src), "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            sys.stderr.write(r.stdout + r.stderr)
            raise RuntimeError(f"hipcc failed on {src}")
        objs.append(obj)
    tmp = LIB + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs, "-lhiprtc"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("link failed")
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
