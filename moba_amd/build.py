"""Builds the HIP kernels into ``moba_amd/libmoba_hip.so`` with hipcc for gfx950, and the extension module
``moba_amd._host`` (csrc/host.cpp, host code) with g++.

Run as ``python -m moba_amd.build``.  hipcc cross-compiles without a GPU.
"""

from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(CSRC, "build")
LIB = os.path.join(HERE, "libmoba_hip.so")
HOST = os.path.join(HERE, "_host" + sysconfig.get_config_var("EXT_SUFFIX"))   # extension module, see csrc/host.cpp
SOURCES = ["chunk_mean.hip", "gate_topk.hip", "lists.hip", "fwd.hip", "fwd_tile.hip", "bwd.hip", "decode.hip", "plan.hip", "probe.hip", "capi.hip"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # packed fp32 instructions stay off: scalar fp32 code only
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument", "-Wno-unknown-warning-option", "-Wno-inline-asm",
]


# per-source extra flags: the attention kernels never produce NaN from finite inputs, and
# telling the compiler so removes the canonicalisation of every MFMA result before a max
EXTRA = {"fwd.hip": ["-fno-honor-nans"], "fwd_tile.hip": ["-fno-honor-nans"]}


def _compile(src: str, force: bool) -> str:
    path = os.path.join(CSRC, src)
    obj = os.path.join(OBJ, src.replace(".hip", ".o"))
    headers = [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".h")]
    deps = [path, *headers, os.path.abspath(__file__)]
    if not force and os.path.exists(obj) and all(os.path.getmtime(obj) > os.path.getmtime(d) for d in deps):
        return obj
    cmd = [HIPCC, *FLAGS, *EXTRA.get(src, []), "-c", path, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr[-8000:]}")
    errs = [l for l in r.stderr.splitlines() if "warning" in l and "packed-fp32-ops" not in l]
    if errs:
        sys.stderr.write("\n".join(errs[:20]) + "\n")
    return obj


def _host_module(force: bool) -> None:
    """csrc/host.cpp against the installed PyTorch (host code only)."""
    import torch
    src = os.path.join(CSRC, "host.cpp")
    deps = [src, os.path.abspath(__file__), os.path.join(os.path.dirname(HERE), "include", "moba_hip.h")]
    root = os.path.dirname(torch.__file__)
    include = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
               os.path.join(os.path.dirname(os.path.dirname(HIPCC)), "include"), sysconfig.get_paths()["include"]]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f'-DMOBA_TORCH_VERSION="{torch.__version__}"',
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *("-I" + d for d in include), src, "-o", HOST,
           "-L" + os.path.join(root, "lib"), "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python"]
    stamp = os.path.join(OBJ, "host.cmd")   # the command the module was built with: PyTorch's version and place are in it
    same = os.path.exists(stamp) and open(stamp).read() == "\n".join(cmd)
    if not force and same and os.path.exists(HOST) and all(os.path.getmtime(HOST) > os.path.getmtime(d) for d in deps):
        return
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed for host.cpp:\n{r.stderr[-8000:]}")
    with open(stamp, "w") as f:
        f.write("\n".join(cmd))
    former = os.path.join(HERE, "_host.so")   # the name without the interpreter's tag that it once had
    if os.path.exists(former):
        os.remove(former)


def build(force: bool = True, verbose: bool = True) -> str:
    os.makedirs(OBJ, exist_ok=True)
    srcs = [s for s in SOURCES if os.path.exists(os.path.join(CSRC, s))]
    with ThreadPoolExecutor(max_workers=min(8, len(srcs) + 1)) as ex:
        host = ex.submit(_host_module, force)
        objs = list(ex.map(lambda s: _compile(s, force), srcs))
        host.result()
    # the hand-issued MFMAs of the dK/dV kernel: nothing touches their results too early in the generated code
    from . import asm_check
    report = asm_check.check_dkv_kernel(asm_check.device_assembly(HIPCC, FLAGS, os.path.join(CSRC, "bwd.hip")))
    if verbose:
        print(report)
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr[-4000:]}")
    if verbose:
        print(f"built {LIB} from {len(objs)} objects")
    return LIB


if __name__ == "__main__":
    build(force="--incremental" not in sys.argv)
