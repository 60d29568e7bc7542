"""Build the gfx950 libraries in-tree.

``libgaudirt_amd.so``: HIP kernels + the C ABI declared in include/gaudirt_amd.h.
``_C*.so``: the PyTorch-ROCm extension (torch.ops.gaudirt.*, PagedMetadata),
linked against libgaudirt_amd.so with an $ORIGIN rpath.

Run ``python -m gaudirt_amd.build`` (or ``__graft_entry__.build()``); every call
recompiles. No GPU is needed: hipcc cross-compiles for gfx950.
"""

import concurrent.futures
import os
import pathlib
import subprocess
import sys
import sysconfig

PACKAGE = pathlib.Path(__file__).resolve().parent
ROOT = PACKAGE.parent
CSRC = PACKAGE / "csrc"
BUILD = PACKAGE / "_build"
ARCH = "gfx950"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

# Packed fp32 VALU forms (v_pk_add/mul/fma_f32) are kept out of generated code:
# some of their forms have given wrong results without an error on this part.
# The host pass warns that it does not know the feature.
DEVICE_FLAGS = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
# Tuning variants of the kernels as extra -D flags, e.g.
# GAUDIRT_AMD_DEFINES="-DGK_STREAM_UNIT_COST=4" (the decode schedule's charge
# per unit); empty for the shipping build.
DEFINES = os.environ.get("GAUDIRT_AMD_DEFINES", "").split()
COMMON = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-I", str(ROOT / "include"), "-I", str(CSRC),
          "-Wall", "-Wno-unused-function", *DEFINES]

LIB_SOURCES = ["gk_api.cpp", "block_allocator_core.cpp", "block_allocator.cpp", "kv_store.hip", "paged_decode.hip", "decode_stream.hip",
               "decode_unit.hip", "paged_prefill.hip", "metadata.hip", "rotary.hip"]
LIB_NAME = "libgaudirt_amd.so"


def _run(cmd):
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(line for line in proc.stdout.splitlines() if "packed-fp32-ops" not in line)
    if proc.returncode != 0:
        raise RuntimeError(f"build step failed ({proc.returncode}): {' '.join(cmd)}\n{out}")
    return out


def _compile(source, extra=()):
    obj = BUILD / (source.replace("/", "_") + ".o")
    src = CSRC / source
    cmd = [HIPCC, *COMMON, *DEVICE_FLAGS, *extra, "-c", str(src), "-o", str(obj)]
    if src.suffix == ".cpp":
        cmd = [HIPCC, *COMMON, *extra, "-x", "hip", "-c", str(src), "-o", str(obj)]
    _run(cmd)
    return obj


def build_library(jobs=8):
    BUILD.mkdir(exist_ok=True)
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as pool:
        objects = list(pool.map(_compile, LIB_SOURCES))
    target = PACKAGE / LIB_NAME
    tmp = target.with_suffix(".so.tmp")
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objects)])
    os.replace(tmp, target)
    return target


def build_extension():
    import torch
    from torch.utils import cpp_extension

    BUILD.mkdir(exist_ok=True)
    includes = []
    for path in cpp_extension.include_paths():
        includes += ["-I", path]
    py_include = sysconfig.get_paths()["include"]
    abi = int(torch._C._GLIBCXX_USE_CXX11_ABI)
    defines = ["-DTORCH_EXTENSION_NAME=_C", "-DTORCH_API_INCLUDE_EXTENSION_H", f"-D_GLIBCXX_USE_CXX11_ABI={abi}",
               "-DUSE_ROCM=1", "-D__HIP_PLATFORM_AMD__=1"]
    src = CSRC / "torch_ext.cpp"
    obj = BUILD / "torch_ext.o"
    _run([HIPCC, "-O2", "-std=c++20", "-fPIC", f"--offload-arch={ARCH}", "-I", str(ROOT / "include"), "-I", str(CSRC),
          "-I", py_include,
          *includes, *defines, "-c", str(src), "-o", str(obj), "-Wno-unused-result"])
    lib_dirs = cpp_extension.library_paths()
    suffix = sysconfig.get_config_var("EXT_SUFFIX")
    target = PACKAGE / f"_C{suffix}"
    tmp = target.with_suffix(".tmp")
    link = [HIPCC, "-shared", "-fPIC", "-o", str(tmp), str(obj), f"-L{PACKAGE}", "-lgaudirt_amd",
            "-Wl,-rpath,$ORIGIN"]
    for d in lib_dirs:
        link += [f"-L{d}", f"-Wl,-rpath,{d}"]
    link += ["-lc10", "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10_hip", "-ltorch_hip"]
    _run(link)
    os.replace(tmp, target)
    return target


def build(jobs=8):
    lib = build_library(jobs)
    ext = build_extension()
    return lib, ext


if __name__ == "__main__":
    for path in build():
        print("built", path)
    sys.exit(0)
