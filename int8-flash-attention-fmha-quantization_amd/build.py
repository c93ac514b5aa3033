"""Build recipe of libfmha_i8.so (one hipcc line, gfx950 only) and of _fmha_torch.so, the host path of the torch entry
points (one g++ line); outputs in-tree beside this file."""
import os
import shutil
import subprocess
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB_PATH = os.path.join(HERE, "libfmha_i8.so")
TORCH_PATH = os.path.join(HERE, "_fmha_torch.so")
TORCH_SOURCE = os.path.join(HERE, "csrc", "fmha_torch.cpp")
SOURCES = [os.path.join(HERE, "csrc", "fmha_i8_api.hip"), os.path.join(HERE, "csrc", "fmha_quant.hip")]
DEPENDS = SOURCES + [os.path.join(HERE, "csrc", "fmha_i8_kernel.hip"),
                     os.path.join(HERE, "csrc", "fmha_i8_split_kernel.hip"),
                     os.path.join(HERE, "csrc", "fmha_i8_pair_kernel.hip"), os.path.join(HERE, "csrc", "fmha_i8_few_kernel.hip"),
                     os.path.join(HERE, "csrc", "fmha_i8_test_builds.h"),
                     os.path.join(HERE, "csrc", "fmha_dequant.h"),
                     os.path.join(ROOT, "include", "fmha_i8.h"), os.path.join(ROOT, "include", "fmha_param_i8.h"),
                     os.path.join(ROOT, "include", "fmha_quant.h")]
# Packed-FP32 instruction selection is switched off for all device code (a flag for hipcc's device pass; the host pass
# prints a harmless "not a recognized feature" note).
HIPCC_FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
               "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
               # MFMA results in ordinary registers: a kernel of one wavefront per SIMD otherwise gets them in accumulation
               # registers and copies every score out of them (a fifth of its instructions)
               "-mllvm", "-amdgpu-mfma-vgpr-form=1"]


def hipcc_path():
    return shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def build_library(verbose=False):
    """Compile the kernel and the C ABI into libfmha_i8.so (always recompiles)."""
    cmd = [hipcc_path()] + HIPCC_FLAGS + ["-I", os.path.join(ROOT, "include"), "-o", LIB_PATH] + SOURCES
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in proc.stdout.splitlines() if "packed-fp32-ops" not in l)
    if proc.returncode != 0:
        raise RuntimeError("hipcc failed:\n" + " ".join(cmd) + "\n" + out)
    if verbose and out.strip():
        print(out)
    return LIB_PATH


def build_torch(verbose=False):
    """Compile the native host path of the torch entry points into _fmha_torch.so (host code only; it calls the C ABI of
    libfmha_i8.so, which must be built first and is found beside it at run time).  None where torch is not installed: the
    library serves C and C++ callers without it."""
    try:
        import torch
    except ImportError:
        print("torch is not installed: %s is not built" % os.path.basename(TORCH_PATH))
        return None
    at = os.path.dirname(torch.__file__)
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(hipcc_path())))
    include = [sysconfig.get_paths()["include"], os.path.join(at, "include"),
               os.path.join(at, "include", "torch", "csrc", "api", "include"), os.path.join(rocm, "include")]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI]
    cmd += [x for d in include for x in ("-I", d)]
    # libfmha_i8.so by name and from this file's own folder, before any LD_LIBRARY_PATH (a library given by its path would be
    # recorded, and looked for, under that path wherever the package goes)
    cmd += ["-o", TORCH_PATH, TORCH_SOURCE, "-L", HERE, "-l:" + os.path.basename(LIB_PATH), "-Wl,-rpath,$ORIGIN",
            "-Wl,--disable-new-dtags", "-L", os.path.join(at, "lib"), "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip",
            "-ltorch_python"]
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if proc.returncode != 0:
        raise RuntimeError("g++ failed:\n" + " ".join(cmd) + "\n" + proc.stdout)
    if verbose and proc.stdout.strip():
        print(proc.stdout)
    return TORCH_PATH


def is_stale():
    if not (os.path.exists(LIB_PATH) and os.path.exists(TORCH_PATH)):
        return True
    t = os.path.getmtime(LIB_PATH)
    return any(os.path.getmtime(p) > t for p in DEPENDS) or os.path.getmtime(TORCH_SOURCE) > os.path.getmtime(TORCH_PATH)


if __name__ == "__main__":
    print(build_library(verbose=True))
    print(build_torch(verbose=True))
