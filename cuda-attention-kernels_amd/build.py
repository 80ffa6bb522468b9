"""Build ``fused_attn/libfused_attn_hip.so`` (and the measurement probe ``fused_attn/libfa_probe.so``)
for gfx950 with hipcc, and the host-only ``fused_attn/libfused_attn_torch.so``, the native dispatcher
kernels of the custom op, against the torch that runs this script.

    python cuda-attention-kernels_amd/build.py          # or __graft_entry__.build()

Each source compiles to an object under ``_build/`` at the repository root, in
parallel, then one shared library is linked next to ``fused_attn/_hip.py`` (the
ctypes loader looks there).  hipcc cross-compiles for gfx950 without a GPU.
"""
from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
BUILD_DIR = os.path.join(ROOT, "_build")
LIB_OUT = os.path.join(HERE, "fused_attn", "libfused_attn_hip.so")
SOURCES = ["fa_prefill.hip", "fa_prefill_f32.hip", "fa_splitk.hip", "fa_generic.hip", "fa_quant.hip", "fa_abi.cpp"]
# the matrix-core ceiling probe bench.py times beside the prefill workload: a library of its own
PROBE_SOURCES = ["fa_ceiling.hip"]
PROBE_OUT = os.path.join(HERE, "fused_attn", "libfa_probe.so")
TORCH_SOURCE = "fa_torch.cpp"
TORCH_OUT = os.path.join(HERE, "fused_attn", "libfused_attn_torch.so")
ARCH = os.environ.get("FUSED_ATTN_ARCH", "gfx950")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
COMMON = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    # no packed-fp32 VALU instructions anywhere in the device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]

# MFMA accumulators in VGPRs for the sources whose D=256 kernels need more than 256 registers: by itself the
# compiler keeps those accumulators in AGPRs and copies them to VGPRs and back around the softmax rescale
# (D=256, B=16 Hq=64 Hkv=8: FP8 decode over 16384 keys 271 -> 234 us; fp32 prefill, 2 x 4 heads, 2048 x 2048:
# 630 -> 601).  The 16-bit prefill keeps the default: it measured 5-7% slower at D=256 with it.
VGPR_FORM = ["-mllvm", "-amdgpu-mfma-vgpr-form=1"]
EXTRA = {"fa_splitk.hip": VGPR_FORM, "fa_prefill_f32.hip": VGPR_FORM}


def _run(cmd: list[str]) -> None:
    r = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(line for line in (r.stdout + r.stderr).splitlines() if noise not in line)
    if r.returncode != 0:
        raise RuntimeError(f"command failed ({r.returncode}): {' '.join(cmd)}\n{err}")
    if err.strip():
        print(err, file=sys.stderr)


def _torch_commands() -> list[list[str]]:
    """Compile and link commands of the dispatcher library."""
    import torch

    root = os.path.dirname(os.path.abspath(torch.__file__))
    inc, lib = os.path.join(root, "include"), os.path.join(root, "lib")
    python = sysconfig.get_paths()["include"]
    rocm = os.path.join(os.path.dirname(os.path.dirname(HIPCC)), "include")
    obj = os.path.join(BUILD_DIR, "fa_torch.o")
    # the build that fused_attn/_hip.py asks for when it loads the library
    build_ = f'-DFA_TORCH_BUILD="{torch.__version__} {torch.version.git_version}"'
    compile_ = [HIPCC, "-x", "c++", "-O2", "-std=c++17", "-fPIC", "-Wall", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM", build_,
                f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-isystem", inc,
                "-isystem", os.path.join(inc, "torch", "csrc", "api", "include"), "-isystem", rocm, "-isystem", python,
                "-c", os.path.join(CSRC, TORCH_SOURCE), "-o", obj]
    link = [HIPCC, "-shared", "-fPIC", obj, "-L", lib, "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip", "-o",
            TORCH_OUT + ".tmp"]
    return [compile_, link]


def _build_torch() -> None:
    for cmd in _torch_commands():
        _run(cmd)
    os.replace(TORCH_OUT + ".tmp", TORCH_OUT)


def build(verbose: bool = False) -> str:
    """Build the libraries.  The dispatcher library is optional (without it calls take the Python path) and needs
    torch's and Python's headers: where it does not build, that is said and the others are built all the same."""
    os.makedirs(BUILD_DIR, exist_ok=True)
    cmds = []

    def objects(sources):
        objs = []
        for src in sources:
            obj = os.path.join(BUILD_DIR, os.path.splitext(src)[0] + ".o")
            cmds.append([HIPCC, *COMMON, *EXTRA.get(src, []), "-x", "hip", "-c", os.path.join(CSRC, src), "-o", obj])
            objs.append(obj)
        return objs

    libs = [(LIB_OUT, objects(SOURCES)), (PROBE_OUT, objects(PROBE_SOURCES))]
    with ThreadPoolExecutor(max_workers=len(cmds) + 1) as ex:
        torch_lib = ex.submit(_build_torch)
        list(ex.map(_run, cmds))
        for out, objs in libs:
            tmp = out + ".tmp"
            _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp])
            os.replace(tmp, out)
            if verbose:
                print(f"built {out}")
        try:
            torch_lib.result()
            if verbose:
                print(f"built {TORCH_OUT}")
        except Exception as e:
            if os.path.exists(TORCH_OUT):  # an older one would not match the sources
                os.remove(TORCH_OUT)
            print(f"{TORCH_OUT} NOT built, attention() takes its slower Python path: {e}", file=sys.stderr)
    return LIB_OUT


if __name__ == "__main__":
    build(verbose=True)
