"""Builds libpicotron_amd.so (the C-ABI library of HIP kernels) and _host.so (the Python extension with the host path of
the hot ops, linked against it) in-tree.

    python -m picotron_amd.build          # compile every csrc/*.hip for gfx950, csrc/host.cpp for the host, and link

hipcc cross-compiles for gfx950 without a GPU present.  Both libraries land next to this file
so that they travel with the source tree; nothing is installed into site-packages.
"""
from __future__ import annotations

import os
import re
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(CSRC, "build")
LIB = os.path.join(HERE, "libpicotron_amd.so")
HOST = os.path.join(HERE, "_host.so")

SOURCES = ["common.hip", "norm.hip", "pointwise.hip", "optim.hip", "loss.hip", "embedding.hip", "product.hip", "product_mid.hip", "product_large.hip", "attn_fwd.hip", "attn_bwd.hip", "attn_bwd_roles.hip"]
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-munsafe-fp-atomics",
    # packed fp32 VALU forms are kept out of the generated code on purpose
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]

# Kernels whose tiles go to LDS without passing the registers, by file and name.  Their dynamic LDS has to start at 0 (no static
# LDS): the requests count their places from there (an address from the compiler is known too late to fold into them, and costs
# an addition per request).  And they wait for a count of their own memory operations: an access to scratch memory would be
# counted with them, and the wait would end before what it waits for is there.
REQUESTING = {"product_mid.hip": "_kernel", "product_large.hip": "_kernel", "attn_fwd.hip": "attn_fwd_kernel",
              "attn_bwd.hip": "dkdv_kernel|dkdv_few_kernel|dq_kernel", "attn_bwd_roles.hip": "roles_kernel"}
RESOURCES = "-Rpass-analysis=kernel-resource-usage"


def kernel_resources(remarks: str) -> dict:
    """{mangled kernel name: {remark: value}} of what the compiler prints with RESOURCES."""
    kernels, now = {}, None
    for key, value in re.findall(r"remark: (?:\S+:\d+:\d+: )?\s*([A-Za-z ]+?)(?: \[[^\]]*\])?: (\S+) \[-Rpass", remarks):
        if key == "Function Name":
            now = kernels.setdefault(value, {})
        else:
            now[key] = int(value) if value.isdigit() else value
    return kernels


def check_requesting(source: str, remarks: str) -> None:
    kernels = {name: r for name, r in kernel_resources(remarks).items() if re.search(REQUESTING[source], name)}
    if not kernels:
        raise RuntimeError(f"{source}: the compiler reported no such kernel's resources")
    for name, r in kernels.items():
        if r["ScratchSize"] or r["VGPRs Spill"] or r["Dynamic Stack"] != "False":
            raise RuntimeError(f"{source}: {name} keeps registers in scratch memory ({r}), and its counted waits would be wrong")
        if r["LDS Size"]:
            raise RuntimeError(f"{source}: {name} has LDS of its own ({r}), and its requests would go there")


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.isabs(cand) and os.path.exists(cand) or not os.path.isabs(cand)):
            return cand
    return "hipcc"


def _run(cmd):
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in proc.stdout.splitlines() if "is not a recognized feature for this target" not in l)
    if proc.returncode != 0:
        raise RuntimeError(f"command failed ({proc.returncode}): {' '.join(cmd)}\n{out}")
    return out


def _compile_host() -> str:
    """csrc/host.cpp -> build/host.o with the host compiler (it holds no device code) against the installed torch."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import COMMON_HIP_FLAGS, include_paths
    obj = os.path.join(OBJ, "host.o")
    includes = [*include_paths(), "/opt/rocm/include", sysconfig.get_paths()["include"]]
    _run(["g++", "-O2", "-std=c++17", *COMMON_HIP_FLAGS, "-DTORCH_EXTENSION_NAME=_host", "-DTORCH_API_INCLUDE_EXTENSION_H",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *[f"-I{d}" for d in includes],
          "-c", os.path.join(CSRC, "host.cpp"), "-o", obj])
    return obj


def _link_host(obj: str) -> str:
    from torch.utils.cpp_extension import library_paths
    dirs = library_paths()
    return _run(["g++", "-shared", "-o", HOST, obj, *[f"-L{d}" for d in dirs], "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10", "-lc10_hip", "-lhipblaslt",
                 f"-L{HERE}", "-lpicotron_amd", "-Wl,-rpath,$ORIGIN"])


def build(verbose: bool = True, extra_flags=()) -> str:
    os.makedirs(OBJ, exist_ok=True)
    hipcc = _hipcc()

    def compile_one(src):
        obj = os.path.join(OBJ, src.replace(".hip", ".o"))
        requesting = src in REQUESTING
        out = _run([hipcc, *FLAGS, *extra_flags, *([RESOURCES] if requesting else []), "-c", os.path.join(CSRC, src), "-o", obj])
        if requesting:
            check_requesting(src, out)
            out = "\n".join(l for l in out.splitlines() if "warning:" in l)   # (of the rest all but warnings are the remarks just read)
        if verbose and out.strip():
            print(out)
        return obj

    with ThreadPoolExecutor(max_workers=8) as pool:
        host = pool.submit(_compile_host)
        objs = list(pool.map(compile_one, SOURCES))
        out = _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB, *objs])
        out += _link_host(host.result())
    if verbose:
        if out.strip():
            print(out)
        print(f"built {LIB} and {HOST}")
    return LIB


if __name__ == "__main__":
    build(extra_flags=tuple(sys.argv[1:]))
