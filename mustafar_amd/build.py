"""Builds libmustafar_hip.so for gfx950 with hipcc (cross-compiles without a GPU), and _host.so beside it."""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libmustafar_hip.so")
HOST = os.path.join(HERE, "_host.so")
SOURCES = ["runtime.hip", "spmv.hip", "compress.hip", "quant.hip", "quant_spmv.hip", "fused.hip", "fused_quant.hip", "window_append.hip"]
# SRAM-ECC on, as it always is on this chip: a load into the upper half of a register then clears the lower half, which gathers
# into the registers of their own addresses rely on (csrc/rank_whole.hpp).  A device without it refuses the library.
ARCH = "gfx950:sramecc+"
FLAGS = [
    "--offload-arch=" + ARCH, "-O3", "-std=c++17", "-fPIC", "-shared",
    # packed-fp32 VALU forms are kept out of the generated code on purpose
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # the leading kernel arguments (up to fourteen 32-bit words) arrive in scalar registers with the wavefront
    # instead of through a load from the argument segment: the first memory round trip of every kernel less
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
    "-Wall", "-Wno-unused-function",
]


def sources():
    return [os.path.join(CSRC, s) for s in SOURCES if os.path.exists(os.path.join(CSRC, s))]


def build(verbose=False):
    """Compiles every source to an object file (in parallel, one hipcc per file) and links the shared library."""
    from concurrent.futures import ThreadPoolExecutor
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    objdir = os.path.join(HERE, "_obj")
    os.makedirs(objdir, exist_ok=True)
    compile_flags = [f for f in FLAGS if f != "-shared"]

    def compile_one(src):
        obj = os.path.join(objdir, os.path.basename(src)[:-4] + ".o")
        cmd = [hipcc] + compile_flags + ["-c", src, "-o", obj]
        if verbose:
            print(" ".join(cmd))
        res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        out = "\n".join(l for l in res.stdout.splitlines() if "packed-fp32-ops" not in l)
        if res.returncode != 0:
            raise RuntimeError("hipcc failed on %s:\n%s" % (src, out))
        return obj, out

    with ThreadPoolExecutor(max_workers=min(8, len(SOURCES))) as pool:
        results = list(pool.map(compile_one, sources()))
    link = [hipcc, "--offload-arch=" + ARCH, "-shared", "-fPIC", "-o", LIB] + [o for o, _ in results]
    res = subprocess.run(link, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if res.returncode != 0:
        raise RuntimeError("link failed:\n" + res.stdout)
    if verbose:
        for _, out in results:
            if out.strip():
                print(out)
    build_host(verbose)
    return LIB


def build_host(verbose=False):
    """The Python module of native calls, by the host compiler against torch's headers and the library above."""
    import sysconfig
    from torch.utils import cpp_extension
    import torch
    libs = os.path.join(os.path.dirname(torch.__file__), "lib")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI]
    cmd += ["-isystem" + p for p in cpp_extension.include_paths()] + ["-I" + sysconfig.get_paths()["include"]]
    cmd += [os.path.join(CSRC, "host.cpp"), "-o", HOST, "-L" + HERE, "-l:libmustafar_hip.so", "-Wl,-rpath,$ORIGIN", "-L" + libs,
            "-lc10", "-ltorch_cpu", "-ltorch_python"]
    if verbose:
        print(" ".join(cmd))
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if res.returncode != 0:
        raise RuntimeError("g++ failed on host.cpp:\n" + res.stdout)


if __name__ == "__main__":
    print(build(verbose=True))
    sys.exit(0)
