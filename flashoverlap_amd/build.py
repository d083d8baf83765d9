"""Build recipe of the native libraries (hipcc, gfx950 only).

  libfo_kernels.so    HIP kernels + host orchestration behind the C ABI of
                      include/flashoverlap.h (no torch dependency)
  libst_pybinding.so  TORCH_LIBRARY shim registering
                      torch.classes.flashoverlap_class.{OverlapImpl,BaselineImpl}
                      and torch.ops.flashoverlap_op.* on top of the C ABI; the
                      file name is the one the reference scripts load
                      (example/RMSNorm.py:5, README.md:69)

  _fo_native.so       Python extension module: the per-call host path of ops.py and
                      layers.py (argument checks, output allocation, one call of the C ABI)

All land in flashoverlap_amd/lib/; the shim is also copied to build/lib/ so that
`torch.ops.load_library("../build/lib/libst_pybinding.so")` keeps working from a
sub-directory of the repository root.

Run as `python -m flashoverlap_amd.build [--no-shim]`.
"""
import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
LIBDIR = os.path.join(PKG, "lib")
OBJDIR = os.path.join(LIBDIR, "obj")
KERNEL_LIB = os.path.join(LIBDIR, "libfo_kernels.so")
SHIM_LIB = os.path.join(LIBDIR, "libst_pybinding.so")
NATIVE_LIB = os.path.join(LIBDIR, "_fo_native.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

KERNEL_SOURCES = ["fo_gemm.hip", "fo_aux.hip", "fo_algo.cpp", "fo_overlap.cpp"]
# fo_gemm256_inst.hip and fo_gemm_tile_inst.hip hold the instantiations of the GEMM kernels for one dtype (fp16 / bf16)
# and one epilogue (plain / signal / scatter / accumulating / reduce-scatter; of the 256x256 kernel also signal / scatter with the
# last wave's sums and the reordered store without counters) per compilation; separate jobs, for a build on many cores.
GEMM_INSTANCES = [(src, d, m) for src in ("fo_gemm256_inst.hip", "fo_gemm_tile_inst.hip") for d in (0, 1) for m in (0, 1, 2, 3, 4)]
GEMM_INSTANCES += [("fo_gemm256_inst.hip", d, m) for d in (0, 1) for m in (5, 6, 7)]

# -packed-fp32-ops off: hipcc must not form v_pk_*_f32 from the float code here.
HIP_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-x", "hip",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # The first fourteen words of a kernel's arguments arrive in scalar registers with the wavefront instead of by a load from
    # memory in front of everything else (whole passes, us: 512x4096x4096 23.25 -> 22.9, 256x1280x3816 13.2 -> 12.9,
    # 2304x1664x912 14.7 -> 14.05, 1152x5120x1720 27.6 -> 26.9).
    "-mllvm", "-amdgpu-kernarg-preload-count=14",
    "-Wno-unused-command-line-argument",
    "-I" + os.path.join(ROOT, "include"), "-I" + CSRC,
]


def _run(cmd):
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if proc.returncode != 0:
        sys.stderr.write(" ".join(cmd) + "\n" + proc.stdout + "\n")
        raise RuntimeError(f"build step failed: {cmd[0]} ... {cmd[-1]}")
    return proc.stdout


def build_kernels(extra_flags=()):
    os.makedirs(OBJDIR, exist_ok=True)

    def compile_one(job):
        src, defs, tag = job
        obj = os.path.join(OBJDIR, os.path.splitext(src)[0] + tag + ".o")
        _run([HIPCC] + HIP_FLAGS + list(extra_flags) + defs + ["-c", os.path.join(CSRC, src), "-o", obj])
        return obj

    # the long jobs first
    jobs = [(src, [f"-DFO_INST_DTYPE={d}", f"-DFO_INST_MODE={m}"], f"_{d}_{m}") for src, d, m in GEMM_INSTANCES]
    jobs += [(src, [], "") for src in KERNEL_SOURCES]
    with ThreadPoolExecutor(max_workers=min(8, os.cpu_count() or 4)) as pool:
        objs = list(pool.map(compile_one, jobs))
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", KERNEL_LIB] + objs)
    return KERNEL_LIB


def _build_torch_lib(src, out, includes=(), libs=()):
    """One g++ source against torch's headers and libraries and libfo_kernels.so."""
    import torch
    from torch.utils import cpp_extension

    os.makedirs(OBJDIR, exist_ok=True)
    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    incs = []
    for p in list(cpp_extension.include_paths()) + list(includes):
        incs += ["-isystem", p]
    abi = int(getattr(torch._C, "_GLIBCXX_USE_CXX11_ABI", True))
    obj = os.path.join(OBJDIR, os.path.splitext(src)[0] + ".o")
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-c", os.path.join(CSRC, src),
          "-o", obj, "-I" + os.path.join(ROOT, "include"), "-isystem", "/opt/rocm/include",
          "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={abi}",
          "-Wno-deprecated-declarations"] + incs)
    _run(["g++", "-shared", "-fPIC", "-o", out, obj,
          "-L" + LIBDIR, "-lfo_kernels", "-Wl,-rpath,$ORIGIN",
          "-L" + torch_lib, *libs, "-ltorch", "-ltorch_cpu", "-lc10", "-ltorch_hip", "-lc10_hip",
          "-Wl,-rpath," + torch_lib,
          "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib"])
    return out


def build_native():
    return _build_torch_lib("fo_native.cpp", NATIVE_LIB, [sysconfig.get_paths()["include"]], ["-ltorch_python"])


def build_shim():
    _build_torch_lib("fo_torch_shim.cpp", SHIM_LIB)
    dst_dir = os.path.join(ROOT, "build", "lib")
    os.makedirs(dst_dir, exist_ok=True)
    # Same directory layout as the reference build output; both libraries are
    # copied so that $ORIGIN resolves the kernel library there too.
    shutil.copy2(SHIM_LIB, os.path.join(dst_dir, "libst_pybinding.so"))
    shutil.copy2(KERNEL_LIB, os.path.join(dst_dir, "libfo_kernels.so"))
    return SHIM_LIB


def build_all(shim=True):
    out = [build_kernels()]
    if shim:
        out += [build_shim(), build_native()]
    return out


if __name__ == "__main__":
    for path in build_all(shim="--no-shim" not in sys.argv):
        print("built", path)
