"""Builds the HIP library and the native host path in-tree.

    python -m simplical_attn_amd.build        # compile every source, link libsa2_hip.so and _sa2_torch.so

One object per .hip file (hipcc for gfx950, compiled in parallel), linked into
simplical_attn_amd/lib/libsa2_hip.so, and csrc/host/sa2_torch.cpp (host code against torch's C++ API) into
simplical_attn_amd/lib/_sa2_torch.so.  Cross-compiles without a GPU.
"""
import concurrent.futures
import glob
import os
import shutil
import subprocess
import sys

from . import listing_check

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
LIB_DIR = os.path.join(PKG, "lib")
LIB_PATH = os.path.join(LIB_DIR, "libsa2_hip.so")
HOST_SRC = os.path.join(CSRC, "host", "sa2_torch.cpp")
HOST_PATH = os.path.join(LIB_DIR, "_sa2_torch.so")
OBJ_DIR = os.path.join(LIB_DIR, "obj")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
# Packed-fp32 VALU forms are switched off for the device pass; the host pass
# does not know the feature and says so, which is harmless.
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-fPIC", "-std=c++17",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    "-I", os.path.join(ROOT, "include"), "-I", CSRC,
]
# sources with hand-placed MFMAs -> their kernels (patterns of the mangled names, ...Li128E...: head_dim 128) and the
# accumulation registers these own (OWNED of their Lone<>); the compiler's listing of them is checked (see listing_check.py)
_KV, _KP = (("mfma_bwd_kv_kernel", 192),), (("mfma_bwd_kp_lone_kernel", 256),)
_SKV, _SKP = (("split_kv_lone_kernel", 192),), (("split_kp_lone_kernel", 256),)
_SFWD = (("split_fwd_lone_kernel.*Li64E", 192), ("split_fwd_lone_kernel.*Li96E", 256))
_FWD = (("mfma_fwd_lone_kernel.*Li64E", 96), ("mfma_fwd_lone_kernel.*Li128E", 192))
HAND_PLACED = {"sa2_mfma_bwd_kv_bf16.hip": _KV, "sa2_mfma_bwd_kv_fp16.hip": _KV,
               "sa2_mfma_bwd_kp_lone_bf16.hip": _KP, "sa2_mfma_bwd_kp_lone_fp16.hip": _KP,
               "sa2_mfma_fwd_lone_bf16.hip": _FWD, "sa2_mfma_fwd_lone_fp16.hip": _FWD,
               "sa2_split_fwd_lone_bf16.hip": _SFWD, "sa2_split_fwd_lone_fp16.hip": _SFWD,
               "sa2_split_fwd_lone_fp32.hip": _SFWD[:1],
               "sa2_split_kp_lone_bf16.hip": _SKP, "sa2_split_kp_lone_fp16.hip": _SKP, "sa2_split_kp_lone_fp32.hip": _SKP,
               "sa2_split_kv_lone_bf16.hip": _SKV, "sa2_split_kv_lone_fp32.hip": _SKV,
               "sa2_split_kv_lone_fp16.hip": (("split_kv_lone_kernel.*Li64E", 192), ("split_kv_lone_kernel.*Li96E", 256))}


def _compile(src, extra):
    name = os.path.basename(src)
    obj = out = os.path.join(OBJ_DIR, name + ".o")
    keep = []
    if name in HAND_PLACED:                    # (the listing is one of the compiler's own steps: kept, no second compilation)
        tmp = os.path.join(OBJ_DIR, name + ".tmp")
        os.makedirs(tmp, exist_ok=True)
        out, keep = os.path.join(tmp, "x.o"), ["-save-temps=obj"]
    res = subprocess.run([HIPCC, *FLAGS, *extra, *keep, "-c", src, "-o", out], capture_output=True, text=True)
    noise = ("is not a recognized feature for this target", "warning generated", "warnings generated")
    err = "\n".join(l for l in res.stderr.splitlines() if not any(n in l for n in noise))
    if res.returncode != 0:
        raise RuntimeError("hipcc failed on %s:\n%s" % (src, err))
    if keep:
        for kernels, owned in HAND_PLACED[name]:
            listing_check.check(glob.glob(os.path.join(tmp, "*gfx950*.s"))[0], kernels, owned)
        os.replace(out, obj)
        shutil.rmtree(tmp)
    return obj, err


def _build_host():
    """The torch extension: no device code, so the host compiler builds it."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension
    inc = [x for d in cpp_extension.include_paths("cuda") if os.path.isdir(d) for x in ("-isystem", d)]
    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    tmp = HOST_PATH + ".tmp"
    cmd = ["g++", "-O2", "-fPIC", "-shared", "-std=c++17", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           "-DTORCH_EXTENSION_NAME=_sa2_torch", "-D_GLIBCXX_USE_CXX11_ABI=%d" % int(torch.compiled_with_cxx11_abi()),
           "-I", os.path.join(ROOT, "include"), *inc, "-isystem", sysconfig.get_paths()["include"], HOST_SRC, "-o", tmp,
           "-L", lib, "-lc10", "-lc10_hip", "-ltorch", "-ltorch_cpu", "-ltorch_python"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("building the host extension failed:\n" + res.stderr)
    os.replace(tmp, HOST_PATH)


def build_library(verbose=True, extra_flags=()):
    os.makedirs(OBJ_DIR, exist_ok=True)
    sources = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, len(sources) + 1)) as ex:
        host = ex.submit(_build_host)
        results = list(ex.map(lambda s: _compile(s, list(extra_flags)), sources))
        host.result()
    for (obj, err), src in zip(results, sources):
        if verbose and err.strip():
            print("[%s]\n%s" % (os.path.basename(src), err), file=sys.stderr)
    objs = [o for o, _ in results]
    tmp = LIB_PATH + ".tmp"
    res = subprocess.run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *objs],
                         capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("link failed:\n" + res.stderr)
    os.replace(tmp, LIB_PATH)
    return LIB_PATH


if __name__ == "__main__":
    print(build_library(extra_flags=sys.argv[1:]))
