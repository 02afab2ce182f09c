"""Builds libbitlinear_hip.so for gfx950 with hipcc, and the CPython module of
host calls (csrc/host_calls.cpp, plain C++ against torch's headers), in-tree.

    python -m bitnet_amd.build

hipcc cross-compiles without a GPU, so this runs anywhere the ROCm toolchain
is installed.  The counterpart of the reference's one-line nvcc recipe
(gpu/bitnet_kernels/compile.sh:1).
"""
import os
import shutil
import subprocess
import sys
import sysconfig

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
REPO_ROOT = os.path.dirname(PKG_DIR)
# source -> extra flags of that translation unit
SOURCES = {
    os.path.join(PKG_DIR, "csrc", "bitlinear_hip.hip"): [],
    os.path.join(PKG_DIR, "csrc", "decoder_ops.hip"): [],
    os.path.join(PKG_DIR, "csrc", "pack.hip"): [],
    os.path.join(PKG_DIR, "csrc", "sample.hip"): [],
    os.path.join(PKG_DIR, "csrc", "decode_stack.hip"): ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
    # keep the attention kernels' accumulators in the vector register file (see the file's header)
    os.path.join(PKG_DIR, "csrc", "attn_prefill.hip"): ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
}
OBJ_DIR = os.path.join(PKG_DIR, "lib", "obj")
LIB_DIR = os.path.join(PKG_DIR, "lib")
LIB_PATH = os.path.join(LIB_DIR, "libbitlinear_hip.so")
HOST_SOURCE = os.path.join(PKG_DIR, "csrc", "host_calls.cpp")
HOST_PATH = os.path.join(LIB_DIR, "_host_calls.so")

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-ffp-contract=off",
    # packed fp32 VALU forms are kept out of all device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # the leading kernel arguments arrive in registers at wave start instead of through scalar loads
    # (a memory round trip in front of every kernel's first useful instruction otherwise)
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
]


def hipcc_path() -> str:
    for cand in (shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found; the HIP library cannot be built")


def _finish(cmd, res, verbose):
    # the host pass warns that it does not know the packed-fp32 feature: harmless
    err = "\n".join(l for l in res.stderr.splitlines() if "packed-fp32-ops" not in l)
    if res.returncode != 0:
        raise RuntimeError("compiler failed: " + " ".join(cmd) + "\n" + res.stdout + err)
    if verbose and err.strip():
        print(err, file=sys.stderr)


def host_command() -> list:
    """The host module's compile line: it holds no device code, so the host compiler builds it."""
    import torch

    root = os.path.dirname(torch.__file__)
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        raise RuntimeError("no host C++ compiler found; the host call module cannot be built")
    inc = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
           os.path.join(os.path.dirname(os.path.dirname(hipcc_path())), "include"), "/opt/rocm/include", sysconfig.get_paths()["include"]]
    abi = int(torch._C._GLIBCXX_USE_CXX11_ABI)
    return [cxx, "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM", f"-D_GLIBCXX_USE_CXX11_ABI={abi}",
            *(f"-I{d}" for d in inc if os.path.isdir(d)), HOST_SOURCE, "-o", HOST_PATH, "-L" + os.path.join(root, "lib"),
            "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch_python"]


def build_library(verbose: bool = True) -> str:
    """One object per source and the host module (compiled side by side), then one link."""
    os.makedirs(OBJ_DIR, exist_ok=True)
    hipcc = hipcc_path()
    host_cmd = host_command()
    if verbose:
        print(" ".join(host_cmd), flush=True)
    host_proc = subprocess.Popen(host_cmd, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)
    jobs = []
    for src, extra in SOURCES.items():
        obj = os.path.join(OBJ_DIR, os.path.splitext(os.path.basename(src))[0] + ".o")
        cmd = [hipcc, *HIPCC_FLAGS, *extra, "-I", os.path.join(REPO_ROOT, "include"), "-c", src, "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        jobs.append((cmd, obj, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)))
    objs = []
    for cmd, obj, proc in jobs:
        out, err = proc.communicate()
        _finish(cmd, subprocess.CompletedProcess(cmd, proc.returncode, out, err), verbose)
        objs.append(obj)
    cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", LIB_PATH]
    if verbose:
        print(" ".join(cmd), flush=True)
    _finish(cmd, subprocess.run(cmd, capture_output=True, text=True), verbose)
    out, err = host_proc.communicate()
    _finish(host_cmd, subprocess.CompletedProcess(host_cmd, host_proc.returncode, out, err), verbose)
    return LIB_PATH


if __name__ == "__main__":
    print(build_library())
