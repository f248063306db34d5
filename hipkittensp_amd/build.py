"""Builds hipkittensp_amd/libmxfp6_gemm.so (gfx950 only) from csrc/*.hip with hipcc, libmxfp6_probes.so beside it, and the
Python binding of the hot calls (_native.so, csrc/binding.cpp) with the host compiler.

    python -m hipkittensp_amd.build            # rebuild everything
The libraries are built in-tree; nothing is installed.  No GPU is needed to build.

libmxfp6_gemm.so is the operator (include/mxfp6_gemm.h).  libmxfp6_probes.so is the measurement build
(include/mxfp6_probes.h): the same objects, except that the C ABI and the e2m3 x e2m3 instantiations of the LDS-tiled
kernel are compiled a second time with -DMXFP6_PROBES (probe entry points, ablation builds, clock stamps) and the probe
kernels (csrc/probes.hip) are added.  bench.py loads it for its ceilings and ablations; the operator never does.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "build")
LIB = os.path.join(HERE, "libmxfp6_gemm.so")
NATIVE = os.path.join(HERE, "_native.so")
PROBES_LIB = os.path.join(HERE, "libmxfp6_probes.so")
SOURCES = ["api.hip", "dispatch.hip", "gemm_generic.hip", "gemm_tiled.hip", "gemm_tiled4.hip", "gemm_block.hip", "gemm_mid.hip", "gemm_skinny.hip", "gemm_ring.hip", "gemm_slice.hip", "quantize.hip"]
# (source, object name, extra flags).  gemm_tiled.hip and gemm_block.hip give five objects each: the host-side part, and the kernel
# instantiations of each pair of operand formats (the bulk of the build time; they compile side by side).  gemm_skinny.hip gives two:
# on packed operands, and on a linear layer's activations.
UNITS = [(src, src.replace(".hip", ""), []) for src in SOURCES] + [
    (f"gemm_{k}.hip", f"gemm_{k}_fmt{fmt}", [f"-DMXFP6_{k.upper()}_FMT={fmt}"]) for k in ("tiled", "block") for fmt in (22, 23, 32, 33)
] + [("gemm_skinny.hip", "gemm_skinny_x", ["-DMXFP6_SKINNY_X"])]
# what the measurement build compiles again (or in addition), with -DMXFP6_PROBES
PROBE_UNITS = [("api.hip", "api_probes", ["-DMXFP6_PROBES"]), ("gemm_tiled.hip", "gemm_tiled_fmt22_probes", ["-DMXFP6_TILED_FMT=22", "-DMXFP6_PROBES"]),
               ("probes.hip", "probes", ["-DMXFP6_PROBES"])]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-std=c++20", "-O3", "-fPIC", "-fvisibility=hidden",
    # packed-fp32 VALU forms are kept out of every kernel of this library
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def _compile(unit) -> str:
    src, name, extra = unit
    obj = os.path.join(OBJ, name + ".o")
    cmd = [HIPCC, *FLAGS, *extra, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode:
        raise RuntimeError(f"hipcc failed on {src} ({name}):\n{err}")
    return obj


def _build_native() -> str:
    """The Python binding of the hot calls: host code against torch's headers, linked to the operator's library beside it."""
    import sysconfig

    import torch

    t = os.path.dirname(torch.__file__)
    cmd = ["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-isystem", os.path.join(t, "include"), "-isystem", "/opt/rocm/include",
           "-isystem", sysconfig.get_paths()["include"], os.path.join(CSRC, "binding.cpp"), "-o", NATIVE,
           "-L", HERE, "-lmxfp6_gemm", "-L", os.path.join(t, "lib"), "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip", "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode:
        raise RuntimeError(f"g++ failed on binding.cpp:\n{r.stderr}")
    return NATIVE


def build(verbose: bool = True) -> str:
    os.makedirs(OBJ, exist_ok=True)
    # the units that take longest first
    order = sorted(UNITS + PROBE_UNITS, key=lambda u: ("_fmt" not in u[1], u[1] not in ("gemm_skinny", "gemm_mid")))
    with cf.ThreadPoolExecutor(max_workers=min(8, len(order))) as ex:
        objs = dict(zip((u[1] for u in order), ex.map(_compile, order)))
    product = [objs[u[1]] for u in UNITS]
    swapped = {"api": "api_probes", "gemm_tiled_fmt22": "gemm_tiled_fmt22_probes"}
    probes = [objs[swapped.get(u[1], u[1])] for u in UNITS] + [objs["probes"]]
    for lib, members in ((LIB, product), (PROBES_LIB, probes)):
        cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", lib, *members]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode:
            raise RuntimeError(f"link failed:\n{r.stderr}")
        if verbose:
            print(f"built {lib}")
    _build_native()
    if verbose:
        print(f"built {NATIVE}")
    return LIB


if __name__ == "__main__":
    build()
    sys.exit(0)
