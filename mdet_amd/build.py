"""Build recipe of the mdet TNF library (libmdet_tnf.so) and its drop-in CLI.

Host C++ is compiled with g++; HIP sources with hipcc for gfx950 only.  Every
HIP compile carries ``-Xclang -target-feature -Xclang -packed-fp32-ops``
(no packed FP32 VALU ops are generated).  Outputs go next to this file:
``mdet_amd/libmdet_tnf.so`` and ``mdet_amd/bin/mdet_tnf_graph``.

Run: ``python -m mdet_amd.build`` (or ``python mdet_amd/build.py``).
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libmdet_tnf.so")
BIN = os.path.join(HERE, "bin", "mdet_tnf_graph")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

HOST_SRCS = ["host_ingest.cpp", "host_gen.cpp", "model_host.cpp", "host_binning.cpp", "host_fit.cpp"]
HIP_SRCS = ["capi_ctx.hip", "tnf_count.hip", "tnf_ingest.hip", "tnf_order.hip", "tnf_pairs.hip", "tnf_ivf.hip", "tnf_mlp.hip", "tnf_fit.hip", "tnf_bin.hip"]

COMMON = ["-O3", "-fPIC", "-std=c++17", "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-Wall"]
HIP_FLAGS = COMMON + [
    "--offload-arch=" + ARCH,
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-fno-gpu-flush-denormals-to-zero",
    "-munsafe-fp-atomics",
]


def _run(cmd):
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if r.returncode != 0:
        raise RuntimeError("build step failed:\n" + " ".join(cmd) + "\n" + r.stdout)
    # keep warnings visible but quiet the known host-pass note about the
    # packed-fp32 target feature
    lines = [ln for ln in r.stdout.splitlines() if "packed-fp32-ops" not in ln and ln.strip()]
    return "\n".join(lines)


def _compile(src):
    path = os.path.join(CSRC, src)
    obj = os.path.join(OBJ, src + ".o")
    if src.endswith(".hip"):
        cmd = [HIPCC] + HIP_FLAGS + ["-c", path, "-o", obj]
    else:
        cmd = ["g++"] + COMMON + ["-pthread", "-c", path, "-o", obj]
    return obj, _run(cmd)


def build(verbose: bool = False) -> str:
    """Compile every source and link libmdet_tnf.so; returns the library path."""
    os.makedirs(OBJ, exist_ok=True)
    srcs = HOST_SRCS + HIP_SRCS
    with ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        results = list(ex.map(_compile, srcs))
    objs = [o for o, _ in results]
    if verbose:
        for (o, msg), s in zip(results, srcs):
            if msg:
                print(f"[{s}]\n{msg}")
    tmp = LIB + ".tmp"
    _run([HIPCC, "--offload-arch=" + ARCH, "-shared", "-fPIC", "-o", tmp] + objs + ["-pthread"])
    os.replace(tmp, LIB)
    # drop-in CLI (C++ over the C ABI, through include/mdet/tnf.hpp)
    cli = os.path.join(CSRC, "tnf_graph_cli.cpp")
    if os.path.exists(cli):
        os.makedirs(os.path.dirname(BIN), exist_ok=True)
        _run(["g++", "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "include"), cli, "-o", BIN,
              "-L" + HERE, "-lmdet_tnf", "-Wl,-rpath,$ORIGIN/..", "-pthread"])
    shutil.rmtree(OBJ, ignore_errors=True)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
