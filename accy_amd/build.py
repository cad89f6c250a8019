"""Builds the gfx950 target in-tree.

* ``accy_amd/_build/libaccy_hip.so`` — the host library behind include/accy_hip.h (C++17, HIP runtime
  and hiprtc). Device code is generated per program and compiled for gfx950 with hiprtc at
  ``accy_hip_compile`` time; the hand-written device sources under ``accy_amd/csrc/kernels/`` are
  embedded into the library as text.
* Each hand-written device source is also compiled with ``hipcc --offload-arch=gfx950`` here, so a
  build on a host without a GPU still checks that every kernel template compiles for CDNA4.
* ``oracle/build/liboracle.so`` — the CPU checker used by tests and bench (not part of the product).
"""
from __future__ import annotations

import os
import subprocess
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent
PKG = ROOT / "accy_amd"
CSRC = PKG / "csrc"
KERNELS = CSRC / "kernels"
BUILD = PKG / "_build"
LIB = BUILD / "libaccy_hip.so"
ORACLE_LIB = ROOT / "oracle" / "build" / "liboracle.so"
ROCM = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))

HOST_SOURCES = ["ir.cpp", "wire.cpp", "lower.cpp", "planner.cpp", "planner_reduce.cpp", "planner_views.cpp",
                "planner_contraction.cpp", "planner_attention.cpp", "runtime.cpp", "tuning.cpp", "tune.cpp", "capi.cpp"]
# Device sources embedded as text: (C++ symbol, file under csrc/kernels).
EMBEDDED = [("kCommonDeviceSource", "common.h"), ("kGemmDeviceSource", "gemm.h"),
            ("kAttentionDeviceSource", "attention.h"), ("kScatterDeviceSource", "scatter.h"),
            ("kDecodeDeviceSource", "decode.h")]
# Packed-f32 instructions stay off in every device build; loops marked `#pragma unroll` unroll
# whatever their size (as for the kernels compiled at run time).
NO_PACKED_F32 = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-mllvm", "-pragma-unroll-threshold=65536"]


def _run(cmd, cwd=None):
    proc = subprocess.run(cmd, cwd=cwd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if proc.returncode != 0:
        sys.stderr.write(proc.stdout)
        raise RuntimeError(f"build step failed: {' '.join(map(str, cmd))}")
    return proc.stdout


def _embed() -> Path:
    out = BUILD / "embedded_sources.cpp"
    parts = ["// Generated by accy_amd/build.py from accy_amd/csrc/kernels: device sources as text.\n",
             "namespace accy {\n"]
    for sym, fname in EMBEDDED:
        path = KERNELS / fname
        text = path.read_text() if path.exists() else ""
        if ")ACCY_SRC\"" in text:
            raise RuntimeError(f"{fname} contains the raw-string delimiter")
        parts.append(f"extern const char* const {sym};\n")
        parts.append(f"const char* const {sym} = R\"ACCY_SRC({text})ACCY_SRC\";\n")
    parts.append("}  // namespace accy\n")
    content = "".join(parts)
    if not out.exists() or out.read_text() != content:
        out.write_text(content)
    return out


def build_scratch_object() -> Path:
    """scratch.hip holds the static device array of the allocation-free entry point; hipcc compiles
    it (host code plus a gfx950 code object holding the array) for linking into the library."""
    obj = BUILD / "scratch.o"
    _run([str(ROCM / "bin" / "hipcc"), "--offload-arch=gfx950", "-O2", "-std=c++17", "-fPIC", *NO_PACKED_F32,
          f"-I{ROOT / 'include'}", "-c", str(CSRC / "scratch.hip"), "-o", str(obj)])
    return obj


def build_library() -> Path:
    BUILD.mkdir(parents=True, exist_ok=True)
    emb = _embed()
    srcs = [str(CSRC / s) for s in HOST_SOURCES] + [str(emb), str(build_scratch_object())]
    cmd = ["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-Wall", "-Wno-unused-function",
           "-D__HIP_PLATFORM_AMD__", f"-I{ROCM / 'include'}", f"-I{ROOT / 'include'}",
           "-o", str(LIB) + ".tmp", *srcs,
           f"-L{ROCM / 'lib'}", "-lamdhip64", "-lhiprtc", f"-Wl,-rpath,{ROCM / 'lib'}"]
    _run(cmd)
    os.replace(str(LIB) + ".tmp", LIB)
    return LIB


def check_device_sources() -> None:
    """Compile each hand-written device source for gfx950 with hipcc (syntax and codegen check)."""
    BUILD.mkdir(parents=True, exist_ok=True)
    for probe in sorted(KERNELS.glob("*_check.hip")):
        obj = BUILD / (probe.stem + ".o")
        _run([str(ROCM / "bin" / "hipcc"), "--offload-arch=gfx950", "-O3", "-std=c++17", *NO_PACKED_F32,
              f"-I{KERNELS}", "-c", str(probe), "-o", str(obj)])


def build_oracle() -> Path:
    _run(["make", "-s", "-C", str(ROOT / "oracle")])
    return ORACLE_LIB


def build_all() -> None:
    build_library()
    check_device_sources()
    build_oracle()


if __name__ == "__main__":
    build_all()
    print(LIB)
