"""Builds libdifflogic_hip.so (the C-ABI kernel library) in-tree with hipcc for gfx950, and _host.so (its callers in C++
that hold torch tensors) with g++.

    python difflogic_amd/build.py
"""
import concurrent.futures
import os
import shutil
import subprocess
import sys
import sysconfig
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")
LIB_NAME = "libdifflogic_hip.so"
LIB_PATH = os.path.join(HERE, LIB_NAME)
SOURCES = ("packed.hip", "lds_net.hip", "train.hip", "schedule.cpp")
# streaming / gather microbenchmarks for `bench.py --ceilings`: a library of their own, never
# loaded by the package
CEILINGS_LIB_PATH = os.path.join(HERE, "libdl_ceilings.so")
CEILINGS_SOURCES = ("ceilings.hip",)

HIPCC_FLAGS = (
    "-O3", "-std=c++17", "--offload-arch=gfx950", "-fPIC", "-shared", "-fvisibility=default",
    # no automatic mul+add fusion: kernels that state the same arithmetic give the same bits
    # (the chained and unchained training kernels are checked for equality); fma is written out
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
)


def hipcc_path():
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (set HIPCC or install ROCm under /opt/rocm)")


# torch tensors and autograd nodes on top of the C ABI
HOST_LIB_PATH = os.path.join(HERE, "_host.so")
HOST_SOURCE = "host.cpp"


def build_library(verbose=False):
    """Compiles every kernel source into one shared library next to this file, the
    measurement helpers into a second one and the native host side into a third."""
    with tempfile.TemporaryDirectory(dir=HERE) as tmp:
        def obj(source):
            return os.path.join(tmp, source + ".o")
        compile_only = [f for f in HIPCC_FLAGS if f != "-shared"]
        commands = [[hipcc_path(), *compile_only, f"-I{INCLUDE}", f"-I{CSRC}", "-c", os.path.join(CSRC, s), "-o", obj(s)]
                    for s in SOURCES + CEILINGS_SOURCES]
        host_compile, host_link = _host_flags()
        commands.append([*host_compile, "-c", os.path.join(CSRC, HOST_SOURCE), "-o", obj(HOST_SOURCE)])
        with concurrent.futures.ThreadPoolExecutor() as pool:
            list(pool.map(lambda cmd: _run(cmd, verbose), commands))
        for sources, out_path in ((SOURCES, LIB_PATH), (CEILINGS_SOURCES, CEILINGS_LIB_PATH)):
            _run([hipcc_path(), *HIPCC_FLAGS, *[obj(s) for s in sources], "-o", out_path + ".tmp"], verbose)
            os.replace(out_path + ".tmp", out_path)
        _run(["g++", "-shared", obj(HOST_SOURCE), *host_link, "-o", HOST_LIB_PATH + ".tmp"], verbose)
        os.replace(HOST_LIB_PATH + ".tmp", HOST_LIB_PATH)
    return LIB_PATH


def _host_flags():
    """Compiler command and link flags for HOST_SOURCE against the torch in this interpreter."""
    import torch
    from torch.utils import cpp_extension
    includes = [INCLUDE, *cpp_extension.include_paths(), os.path.join(cpp_extension.ROCM_HOME or "/opt/rocm", "include"),
                sysconfig.get_paths()["include"]]
    compile_ = ["g++", "-O2", "-std=c++17", "-fPIC", "-DTORCH_EXTENSION_NAME=_host", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
                f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *[f"-I{p}" for p in includes]]
    link = [f"-L{HERE}", "-ldifflogic_hip", *[f"-L{p}" for p in cpp_extension.library_paths()], "-lc10", "-ltorch", "-ltorch_cpu",
            "-ltorch_python", "-lc10_hip", "-ltorch_hip", "-Wl,-rpath,$ORIGIN"]
    return compile_, link


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    # hipcc's host pass warns that it does not know the packed-fp32 feature; that is expected.
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in proc.stderr.splitlines() if noise not in l)
    if proc.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed ({proc.returncode}):\n{err}")
    if verbose and err.strip():
        print(err, file=sys.stderr)


if __name__ == "__main__":
    print(build_library(verbose=True))
