"""Build recipe of the native library ``libullm_hip.so`` (gfx950 only).

Every HIP source is compiled by hipcc for ``--offload-arch=gfx950`` with
packed-FP32 instruction selection disabled and IEEE fp32 division, then linked
into one shared library exporting the C ABI of include/ullm/*.h.  The library
is built in-tree (``ullm-project_amd/lib``) so that it travels with the tree.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "src"
BUILD = PKG / "_build"
LIB = PKG / "lib" / "libullm_hip.so"
# Measurement aid of bench.py (a streaming-read floor kernel); not linked
# into the product library.
BENCH_LIB = PKG / "lib" / "libullm_bench.so"
BENCH_SOURCES = ["bench_read.hip", "check_bf16.hip"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SOURCES = ["abi_v1.cpp", "linear_api.cpp", "safetensors.cpp", "evidence.hip", "noalloc.hip", "weights.hip",
           "gemv.hip", "gemm_wq.hip", "gemm_fp8.hip"]

COMMON = [
    "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden",
    "--offload-arch=gfx950",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-fno-gpu-flush-denormals-to-zero",
    "-Wall", "-Wextra", "-Wno-unused-parameter",
    f"-I{ROOT / 'include'}", f"-I{CSRC}",
]


def _compile(src: str) -> Path:
    out = BUILD / (src + ".o")
    cmd = [HIPCC, *COMMON, "-x", "hip", "-c", str(CSRC / src), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr}")
    if r.stderr.strip():
        # warnings other than the known host-side packed-fp32 notice
        lines = [l for l in r.stderr.splitlines()
                 if "packed-fp32-ops" not in l and l.strip()]
        if lines:
            sys.stderr.write("\n".join(lines) + "\n")
    return out


CMAKE_BUILD = BUILD / "cmake"
ARCHIVE = CMAKE_BUILD / "libullm_hip_stub.a"
# A C program linked against the static archive (tests/archive_check.c), run
# by tests/test_gpu_archive.py on the GPU box.
ARCHIVE_CHECK = PKG / "lib" / "ullm_archive_check"


def build_static() -> Path:
    """Build the CMake project's static target ullm_hip_stub with the
    arguments the reference's ullm-hip-sys build.rs passes, and link
    tests/archive_check.c against it as a Rust binary would link the crate
    (the archive, amdhip64, stdc++)."""
    rocm = Path("/opt/rocm")
    subprocess.run(
        ["cmake", "-S", str(PKG), "-B", str(CMAKE_BUILD), "-G", "Unix Makefiles",
         "-DCMAKE_BUILD_TYPE=release", f"-DCMAKE_ARCHIVE_OUTPUT_DIRECTORY={CMAKE_BUILD}",
         f"-DROCM_PATH={rocm}", f"-DCMAKE_HIP_COMPILER={rocm}/bin/amdclang++",
         "-DCMAKE_HIP_ARCHITECTURES=gfx950", "-DULLM_HIP_COMPILE_TARGET=gfx950",
         "-DULLM_ENABLE_HIP_COMPILE_PROBE=OFF", "-DULLM_ENABLE_HIP_RUNTIME=ON"],
        check=True, capture_output=True, text=True)
    r = subprocess.run(["cmake", "--build", str(CMAKE_BUILD), "--target", "ullm_hip_stub",
                        "-j8"], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"cmake build of ullm_hip_stub failed:\n{r.stdout[-4000:]}{r.stderr[-4000:]}")
    tmp = ARCHIVE_CHECK.with_suffix(".tmp")
    subprocess.run(
        ["gcc", "-std=c11", "-O2", "-Wall", "-Wextra", "-Werror", "-D__HIP_PLATFORM_AMD__",
         f"-I{ROOT / 'include'}", f"-I{rocm / 'include'}", str(ROOT / "tests" / "archive_check.c"),
         f"-L{CMAKE_BUILD}", "-lullm_hip_stub", f"-L{rocm / 'lib'}", "-lamdhip64", "-lstdc++",
         "-lm", f"-Wl,-rpath,{rocm / 'lib'}", "-o", str(tmp)], check=True)
    os.replace(tmp, ARCHIVE_CHECK)
    return ARCHIVE


def build() -> Path:
    """Compile every source (always) and link libullm_hip.so."""
    BUILD.mkdir(exist_ok=True)
    LIB.parent.mkdir(exist_ok=True)
    with ThreadPoolExecutor(max_workers=min(8, len(SOURCES) + len(BENCH_SOURCES))) as ex:
        objs = list(ex.map(_compile, SOURCES + BENCH_SOURCES))
    for lib, n in ((LIB, len(SOURCES)), (BENCH_LIB, None)):
        parts = objs[:n] if n is not None else objs[len(SOURCES):]
        tmp = lib.with_suffix(".so.tmp")
        cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC",
               *map(str, parts), "-o", str(tmp)]
        subprocess.run(cmd, check=True)
        os.replace(tmp, lib)
    return LIB


if __name__ == "__main__":
    print(build())
