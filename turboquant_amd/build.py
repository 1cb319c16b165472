"""Compile the HIP sources under csrc/ into turboquant_amd/libtq_hip.so for gfx950.

hipcc cross-compiles without a GPU, so this runs in the build container; the
shared object is loaded by `_ffi.py` and is never built implicitly at import.
"""

from __future__ import annotations

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libtq_hip.so")
HOST = os.path.join(HERE, "_tq_host.so")           # (imported by _ffi.py, where it fits the torch that runs)
# (the matrix-core page kernel is instantiated by one file per head size, so that they compile side by side)
SOURCES = ["tq_decode_mfma_d128.hip", "tq_decode_mfma_d128_f16.hip", "tq_decode_mfma_d64.hip", "tq_decode_mfma_d64_f16.hip",
           "tq_decode_mfma_d256.hip", "tq_quantize_mfma.hip", "tq_quantize_wide.hip", "tq_decode_wide.hip", "tq_decode_heads.hip",
           "tq_quantize.hip", "tq_score.hip", "tq_decode.hip", "tq_decode_mfma.hip", "tq_probe.hip"]

# packed-fp32 instructions stay off: some of their forms have produced wrong
# results on this hardware pool
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # no implicit a*b+c fusion: the quantisers mirror separately rounded torch ops;
    # the kernels call fmaf() explicitly wherever a fused multiply-add is wanted
    "-ffp-contract=off",
    # the first 14 argument dwords of a kernel arrive in registers: a launch does not begin with a memory latency
    # (14 decode steps of 24 - 72 us: 0.1 - 0.5 us each; 16 x 8192 tokens, 32 q / 8 KV heads of 128: 38.7 -> 38.6)
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
    "-fno-gpu-rdc", "-Wall", "-Wno-unused-function",
    # the LDS-direct loads name m0 in their clobber lists, which the compiler reports as a reserved register
    "-Wno-inline-asm",
]


def _run(cmd):
    try:
        res = subprocess.run(cmd, capture_output=True, text=True)
    except OSError as e:                       # (no such compiler)
        return 127, str(e)
    # the host pass warns that it does not know the packed-fp32 feature; that is harmless
    err = "\n".join(l for l in res.stderr.splitlines() if "packed-fp32-ops" not in l)
    return res.returncode, err


def _host_command(out):
    """The native host side of small calls: a Python module against torch's headers, no device code."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths

    from ._ffi import host_stamp
    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    # NDEBUG: without it pybind11 keeps a thread-local count of references, and a module with thread-local data that is loaded behind
    # libtq_hip.so slows the lookup of that library's own, about 1 us per launch (a ragged write of 3 short prompts 10.0 -> 11.4 us)
    headers = [*include_paths(), sysconfig.get_paths()["include"], "/opt/rocm/include"]
    return ([os.environ.get("CXX", "g++"), "-O2", "-DNDEBUG", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
             f'-DTQ_HOST_STAMP="{host_stamp()}"',
             f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}"] + [x for h in headers for x in ("-isystem", h)] +
            [os.path.join(CSRC, "tq_host.cpp"), "-L" + lib] + [f"-l{n}" for n in ("c10", "c10_hip", "torch_cpu", "torch_hip", "torch", "torch_python")] +
            ["-o", out])


def _build_host(out):
    """(status, messages) of the native host side, compiled to `out`: it needs more than hipcc (g++, torch's and Python's headers)."""
    try:
        return _run(_host_command(out))
    except Exception as e:
        return 1, f"{type(e).__name__}: {e}"


def build_library(verbose: bool = False) -> str:
    """Compile every source to an object file (in parallel: the files are independent translation units)
    and link them into libtq_hip.so; with it the native host side of small calls, which the package does without where it does not
    compile (it takes the place of the former one once the library stands, and the former one does not stay behind)."""
    from concurrent.futures import ThreadPoolExecutor
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    objdir = os.path.join(HERE, "build")
    os.makedirs(objdir, exist_ok=True)
    # TQ_EXTRA_HIPCC_FLAGS: extra compile flags, e.g. -DTQ_STAMPS for the page kernel's phase time stamps
    compile_flags = [f for f in FLAGS if f != "-shared"] + os.environ.get("TQ_EXTRA_HIPCC_FLAGS", "").split()
    jobs = []
    for src in SOURCES:
        obj = os.path.join(objdir, src.replace(".hip", ".o"))
        jobs.append((obj, [hipcc] + compile_flags + ["-c", os.path.join(CSRC, src), "-o", obj]))
    host_built = os.path.join(objdir, os.path.basename(HOST))
    if verbose:
        for _, cmd in jobs:
            print(" ".join(cmd))
    with ThreadPoolExecutor(max_workers=min(len(jobs) + 1, os.cpu_count() or 1)) as pool:
        host = pool.submit(_build_host, host_built)
        results = list(pool.map(lambda j: _run(j[1]), jobs))
        host_rc, host_err = host.result()
    for (obj, _), (rc, err) in zip(jobs, results):
        if rc != 0:
            raise RuntimeError(f"hipcc failed ({rc}) for {obj}:\n{err}")
        if verbose and err.strip():
            print(err, file=sys.stderr)
    link = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-fno-gpu-rdc"] + [obj for obj, _ in jobs] + ["-o", LIB]
    if verbose:
        print(" ".join(link))
    rc, err = _run(link)
    if rc != 0:
        raise RuntimeError(f"hipcc link failed ({rc}):\n{err}")
    if host_rc == 0:
        os.replace(host_built, HOST)
    else:
        print(f"warning: the native host side is not built ({host_rc}), small calls take longer on the host:\n{host_err}", file=sys.stderr)
        if os.path.exists(HOST):
            os.remove(HOST)
    return LIB


if __name__ == "__main__":
    print(build_library(verbose=True))
