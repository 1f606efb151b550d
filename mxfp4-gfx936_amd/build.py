"""Build libmxfp4_gfx950.so for MI355X (gfx950) in-tree.

``python mxfp4-gfx936_amd/build.py`` compiles every ``csrc/*.hip`` with
hipcc (in parallel, objects under ``_build/``) and links
``mxfp4_amd/libmxfp4_gfx950.so`` next to the Python package that loads it,
and ``mxfp4_amd/libmxfp4_probe.so`` (``csrc/probe/``: a plain HBM read that
bench.py times as the floor of the decode kernels; not part of the library),
and with the host compiler ``mxfp4_amd/_host.so`` (``host/``: the operators'
plain calls, against the installed torch).

Flags: ``-O3`` for gfx950 only; packed-FP32 instruction selection is turned
off (``-Xclang -target-feature -Xclang -packed-fp32-ops``); denormals are
kept (no fast-math / flush-to-zero), which the bit-exact dequant and the
subnormal E8M0 scale (s = 0 -> 2^-127) rely on.
"""

from __future__ import annotations

import concurrent.futures as cf
import glob
import os
import re
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")
OBJ_DIR = os.path.join(HERE, "_build")
GEN_DIR = os.path.join(OBJ_DIR, "gen")  # generated sources (silu_table.inc)
LIB = os.path.join(HERE, "mxfp4_amd", "libmxfp4_gfx950.so")
# measurement aid for bench.py (a plain HBM read), kept out of the library
PROBE_SRC = os.path.join(CSRC, "probe", "read_floor.hip")
PROBE_LIB = os.path.join(HERE, "mxfp4_amd", "libmxfp4_probe.so")
# the operators' plain calls in native code (torch's C++ interface)
HOST_SRC = os.path.join(HERE, "host", "mxfp4_host.cpp")
HOST_LIB = os.path.join(HERE, "mxfp4_amd", "_host.so")
CXX = os.environ.get("CXX", "g++")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

CFLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    f"-I{INCLUDE}",
    f"-I{GEN_DIR}",
]


# kernels whose waits count loads, with no room for scratch accesses: the build
# fails if the compiler spills in one
NO_SCRATCH = ("gemm_w4a16_dr.hip",)
_RESOURCES = "-Rpass-analysis=kernel-resource-usage"


def check_no_scratch(src: str, remarks: str) -> None:
    """RuntimeError unless the compiler's resource remarks report kernels, all
    without scratch."""
    names = re.findall(r"remark: +Function Name: (\S+)", remarks)
    sizes = [int(v) for v in re.findall(r"remark: +ScratchSize \[bytes/lane\]: (\d+)", remarks)]
    if not names or len(names) != len(sizes):
        raise RuntimeError(f"{src}: no resource usage reported")
    bad = [f"{n} ({v} bytes/lane)" for n, v in zip(names, sizes) if v]
    if bad:
        raise RuntimeError(f"{src}: scratch in " + ", ".join(bad))


def _compile(src: str, verbose: bool) -> str:
    obj = os.path.join(OBJ_DIR, os.path.basename(src) + ".o")
    no_scratch = os.path.basename(src) in NO_SCRATCH
    cmd = [HIPCC, *CFLAGS, *([_RESOURCES] if no_scratch else []), "-c", src, "-o", obj]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    # hipcc's host pass does not know the packed-fp32 feature and says so;
    # that line is expected, anything else is shown.
    noise = "is not a recognized feature for this target"
    msgs = [ln for ln in (res.stdout + res.stderr).splitlines() if noise not in ln]
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n" + "\n".join(msgs))
    if no_scratch:
        check_no_scratch(src, res.stdout + res.stderr)
    if msgs and verbose:
        print("\n".join(msgs), flush=True)
    return obj


def _build_host(verbose: bool) -> None:
    """The CPython module ``mxfp4_amd/_host.so`` against the installed torch
    (optional: without it the operators call the library from Python)."""
    import sysconfig

    try:
        import torch
        from torch.utils import cpp_extension
    except ImportError as e:
        print(f"torch cannot be imported ({e}): _host.so is not built", flush=True)
        return
    version = f"{torch.__version__} {torch.version.git_version}"  # as _lib.torch_build
    root = os.path.dirname(torch.__file__)
    libs = os.path.join(root, "lib")
    incs = [*cpp_extension.include_paths(), os.path.join(os.path.dirname(os.path.dirname(HIPCC)),
                                                         "include"),
            sysconfig.get_paths()["include"], INCLUDE]
    tmp = HOST_LIB + ".tmp"
    cmd = [CXX, "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f'-DMXFP4_TORCH="{version}"',
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *[f"-isystem{i}" for i in incs], HOST_SRC, f"-L{libs}", "-ltorch_python", "-ltorch",
           "-ltorch_cpu", "-lc10", "-lc10_hip", f"-Wl,-rpath,{libs}", "-o", tmp]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{CXX} failed for {HOST_SRC}:\n{res.stdout}{res.stderr}")
    os.replace(tmp, HOST_LIB)


def build(verbose: bool = False) -> str:
    """Compile all HIP sources and link the shared library; returns its path."""
    os.makedirs(GEN_DIR, exist_ok=True)
    sys.path.insert(0, HERE)
    import silu_table  # the SiLU lookup tables of csrc/silu.h
    silu_table.write_inc(os.path.join(GEN_DIR, "silu_table.inc"))
    sources = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    if not sources:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    workers = min(len(sources) + 1, max(1, min(8, os.cpu_count() or 1)))
    with cf.ThreadPoolExecutor(workers) as ex:
        host = ex.submit(_build_host, verbose)
        objs = list(ex.map(lambda s: _compile(s, verbose), sources))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    os.replace(tmp, LIB)
    tmp = PROBE_LIB + ".tmp"
    cmd = [HIPCC, *CFLAGS, "-shared", PROBE_SRC, "-o", tmp]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {PROBE_SRC}:\n{res.stdout}{res.stderr}")
    os.replace(tmp, PROBE_LIB)
    host.result()  # raises what it raised, with the library in place
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
