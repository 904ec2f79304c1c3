"""Build libtension_hip.so for gfx950 with hipcc (no GPU needed).

    python -m bozo_amd.build          # always recompiles

Each HIP translation unit is compiled in parallel to an object file under
bozo_amd/_build/, then linked into bozo_amd/lib/libtension_hip.so.  The eager
call path (csrc/host.cpp, host code only) is compiled with the C++ compiler
against the installed torch and linked to that library: bozo_amd/lib/_host.so.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
import sysconfig

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
INCLUDE = os.path.join(ROOT, "include")
OBJDIR = os.path.join(PKG, "_build")
LIBDIR = os.path.join(PKG, "lib")
LIBNAME = "libtension_hip.so"
HOSTNAME = "_host.so"
ARCH = os.environ.get("TENSION_OFFLOAD_ARCH", "gfx950")

SOURCES = [
    "capi.hip", "exact.hip", "decode.hip",
    "mfma.hip", "mfma_fwd.hip", "mfma_dq.hip", "mfma_dkv.hip", "mfma_bwd_fused.hip", "mfma_global.hip",
    "mfma_wide.hip",
    "split.hip", "split_fwd_bf16.hip", "split_dq_bf16.hip", "split_dkv_bf16.hip",
    "split_fwd_f32.hip", "split_dq_f32.hip", "split_dkv_f32.hip",
    "split_fwd_f32v.hip", "split_dq_f32v.hip", "split_dkv_f32v.hip",
    "split_fwd_f16.hip", "split_dq_f16.hip", "split_dkv_f16.hip",
    "tau_export.hip", "graph_bias.hip", "aux_loss.hip",
    "exact_fwd_f32.hip", "exact_dq_f32.hip", "exact_dkv_f32.hip",
    "exact_fwd_f64.hip", "exact_dq_f64.hip", "exact_dkv_f64.hip",
]

HIPCC_FLAGS = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
    # code-object v5 loads under both torch's bundled HIP 7.0 runtime and /opt/rocm 7.2
    "-mcode-object-version=5",
    # no packed-fp32 VALU instructions in device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (ROCm toolchain required to build libtension_hip.so)")


def _compile(src: str) -> str:
    obj = os.path.join(OBJDIR, os.path.splitext(src)[0] + ".o")
    cmd = [hipcc(), *HIPCC_FLAGS, "-I", INCLUDE, "-I", CSRC, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{r.stdout}\n{r.stderr}")
    # the host pass prints a harmless notice about the device-only feature flag
    noise = "packed-fp32-ops' is not a recognized feature"
    msgs = [ln for ln in (r.stderr or "").splitlines() if noise not in ln and ln.strip()]
    if msgs:
        sys.stderr.write("\n".join(msgs) + "\n")
    return obj


def _host_compile() -> str:
    import torch
    from torch.utils import cpp_extension
    obj = os.path.join(OBJDIR, "host.o")
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-Wall",
           "-DTORCH_EXTENSION_NAME=_host", "-DTORCH_API_INCLUDE_EXTENSION_H", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-I", INCLUDE]
    for d in [*cpp_extension.include_paths("cuda"), sysconfig.get_paths()["include"]]:
        cmd += ["-isystem", d]
    r = subprocess.run(cmd + ["-c", os.path.join(CSRC, "host.cpp"), "-o", obj], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed on host.cpp:\n{r.stdout}\n{r.stderr}")
    return obj


def _host_link(obj: str) -> None:
    from torch.utils import cpp_extension
    out = os.path.join(LIBDIR, HOSTNAME)
    cmd = [os.environ.get("CXX", "g++"), "-shared", obj, "-o", out + ".tmp",
           *[f"-L{d}" for d in cpp_extension.library_paths("cuda")], "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch",
           "-ltorch_python", f"-L{LIBDIR}", f"-l:{LIBNAME}", "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link of {HOSTNAME} failed:\n{r.stdout}\n{r.stderr}")
    os.replace(out + ".tmp", out)


def build(verbose: bool = True) -> str:
    os.makedirs(OBJDIR, exist_ok=True)
    os.makedirs(LIBDIR, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=min(len(SOURCES), os.cpu_count() or 4, 16)) as ex:
        host = ex.submit(_host_compile)
        objs = list(ex.map(_compile, SOURCES))
        host_obj = host.result()
    out = os.path.join(LIBDIR, LIBNAME)
    tmp = out + ".tmp"
    cmd = [hipcc(), "-shared", "-fPIC", f"--offload-arch={ARCH}", *objs, "-o", tmp]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, out)
    _host_link(host_obj)
    if verbose:
        print(f"built {out}")
    return out


if __name__ == "__main__":
    build()
