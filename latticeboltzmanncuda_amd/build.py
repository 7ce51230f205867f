"""Build recipe for the native libraries (gfx950 HIP + host C++).

    python -m latticeboltzmanncuda_amd.build

produces, in-tree under latticeboltzmanncuda_amd/lib/:
  liblbm_hip.so   the C-ABI of include/lbm.h (HIP kernels for gfx950)
  liblbm.so       the host-only C++ facade of include/lbm/*.h (Lattice,
                  Model, Geometry, FlowData ...) over that C-ABI (g++)
and under latticeboltzmanncuda_amd/bin/ the C++ test suites of tests/cpp/
and the command-line driver LatticeBoltzmannHip (cli/).

Every .hip file is compiled to an object with hipcc (parallel), then
linked into one shared library.  Compilation always runs (no staleness
check), so a call after a source change always rebuilds.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
HOST = os.path.join(PKG, "host")
LIBDIR = os.path.join(PKG, "lib")
OBJDIR = os.path.join(PKG, "lib", "obj")
INCLUDE = os.path.join(ROOT, "include")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
HIP_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Wno-unused-function",
    # keep packed-FP32 instructions out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    f"-I{INCLUDE}",
]

HIP_SOURCES = ["lbm_capi.hip", "k_standard.hip", "k_reference.hip",
               "k_common.hip", "lbm_batch.hip", "k_batch.hip",
               "lbm_serve.hip", "k_voxel.hip", "k_receivers.hip",
               "lbm_snapshot.hip",
               "lbm_exports.hip", "lbm_noalloc.hip", "lbm_transfer.hip"]
HOST_SOURCES = ["Constants.cpp", "Geometry.cpp", "Utils.cpp",
                "FlowCriterion.cpp", "Model.cpp", "Lattice.cpp"]
CXX = os.environ.get("CXX", "g++")
# portable x86-64 code: the library is built here and runs on the GPU host
CXX_FLAGS = ["-O2", "-std=c++17", "-fPIC", "-fopenmp", "-march=x86-64-v2",
             "-Wall", f"-I{INCLUDE}", f"-I{os.path.join(INCLUDE, 'lbm')}"]
BINDIR = os.path.join(PKG, "bin")
TESTS_CPP = os.path.join(ROOT, "tests", "cpp")
CPP_SUITES = ["GeometryTest", "ModelTest", "CalculationsTest",
              "CoordinatesTest", "GeometryDump"]


def _run(cmd: list[str]) -> None:
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                       text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout)
        raise RuntimeError("build step failed: " + " ".join(cmd))
    # surface real warnings, drop the host pass's note about the GPU-only
    # target feature
    lines = [l for l in r.stdout.splitlines()
             if "packed-fp32-ops" not in l and l.strip()]
    if lines:
        sys.stderr.write("\n".join(lines) + "\n")


def _compile_hip(src: str) -> str:
    obj = os.path.join(OBJDIR, os.path.splitext(src)[0] + ".o")
    _run([HIPCC, *HIP_FLAGS, "-c", os.path.join(CSRC, src), "-o", obj])
    return obj


def build_hip(jobs: int | None = None) -> str:
    os.makedirs(OBJDIR, exist_ok=True)
    jobs = jobs or min(len(HIP_SOURCES), os.cpu_count() or 4)
    with cf.ThreadPoolExecutor(jobs) as ex:
        objs = list(ex.map(_compile_hip, HIP_SOURCES))
    out = os.path.join(LIBDIR, "liblbm_hip.so")
    tmp = out + ".tmp"
    # roctx ranges (rocprofiler-sdk) mark step and serving chunks for
    # rocprofv3 --marker-trace
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs,
          "-L/opt/rocm/lib", "-lrocprofiler-sdk-roctx", "-Wl,-rpath,/opt/rocm/lib",
          "-o", tmp])
    os.replace(tmp, out)
    return out


def build_facade() -> str:
    """liblbm.so: the C++ facade, linked against liblbm_hip.so."""
    os.makedirs(OBJDIR, exist_ok=True)
    objs = []
    for src in HOST_SOURCES:
        obj = os.path.join(OBJDIR, "host_" + os.path.splitext(src)[0] + ".o")
        objs.append(obj)
    with cf.ThreadPoolExecutor(len(HOST_SOURCES)) as ex:
        list(ex.map(lambda so: _run([CXX, *CXX_FLAGS, "-c",
                                     os.path.join(HOST, so[0]), "-o", so[1]]),
                    zip(HOST_SOURCES, objs)))
    out = os.path.join(LIBDIR, "liblbm.so")
    tmp = out + ".tmp"
    _run([CXX, "-shared", "-fopenmp", *objs, f"-L{LIBDIR}", "-llbm_hip",
          "-Wl,-rpath,$ORIGIN", "-o", tmp])
    os.replace(tmp, out)
    return out


def build_cpp_suites() -> list[str]:
    """The C++ suites of tests/cpp (the reference's four gtest suites
    re-expressed on the facade)."""
    os.makedirs(BINDIR, exist_ok=True)

    def one(name: str) -> str:
        out = os.path.join(BINDIR, name)
        _run([CXX, *CXX_FLAGS, f"-I{TESTS_CPP}",
              os.path.join(TESTS_CPP, name + ".cpp"), f"-L{LIBDIR}", "-llbm",
              "-llbm_hip", "-Wl,-rpath,$ORIGIN/../lib", "-o", out + ".tmp"])
        os.replace(out + ".tmp", out)
        return out

    with cf.ThreadPoolExecutor(len(CPP_SUITES)) as ex:
        return list(ex.map(one, CPP_SUITES))


CLI_DIR = os.path.join(PKG, "cli")


def build_cli() -> str:
    """bin/LatticeBoltzmannHip: the reference's command-line driver on the
    facade."""
    os.makedirs(BINDIR, exist_ok=True)
    out = os.path.join(BINDIR, "LatticeBoltzmannHip")
    _run([CXX, *CXX_FLAGS, os.path.join(CLI_DIR, "LatticeBoltzmannHip.cpp"),
          f"-L{LIBDIR}", "-llbm", "-llbm_hip", "-Wl,-rpath,$ORIGIN/../lib",
          "-o", out + ".tmp"])
    os.replace(out + ".tmp", out)
    return out


SAN_FLAGS = ["-O1", "-g", "-fno-omit-frame-pointer",
             "-fsanitize=address,undefined", "-fno-sanitize-recover=all"]


def build_sanitized() -> list[str]:
    """The host facade (host/*.cpp) and the C++ suites of tests/cpp built by
    g++ under AddressSanitizer and UndefinedBehaviorSanitizer, every report
    fatal: lib_san/liblbm.so and bin_san/<suite>.  They link the ordinary
    liblbm_hip.so (the HIP layer is not instrumented; the suites the CPU
    tests run make no GPU call).  tests/run_sanitized.sh runs the CPU tests
    on them."""
    libdir = os.path.join(PKG, "lib_san")
    bindir = os.path.join(PKG, "bin_san")
    objdir = os.path.join(libdir, "obj")
    os.makedirs(objdir, exist_ok=True)
    os.makedirs(bindir, exist_ok=True)
    flags = [f for f in CXX_FLAGS if f != "-O2"] + SAN_FLAGS
    objs = [os.path.join(objdir, os.path.splitext(s)[0] + ".o")
            for s in HOST_SOURCES]
    with cf.ThreadPoolExecutor(len(HOST_SOURCES)) as ex:
        list(ex.map(lambda so: _run([CXX, *flags, "-c", os.path.join(HOST, so[0]),
                                     "-o", so[1]]),
                    zip(HOST_SOURCES, objs)))
    lib = os.path.join(libdir, "liblbm.so")
    _run([CXX, "-shared", "-fopenmp", *SAN_FLAGS, *objs, f"-L{LIBDIR}",
          "-llbm_hip", f"-Wl,-rpath,{LIBDIR}", "-o", lib + ".tmp"])
    os.replace(lib + ".tmp", lib)

    def one(name: str) -> str:
        out = os.path.join(bindir, name)
        _run([CXX, *flags, f"-I{TESTS_CPP}", os.path.join(TESTS_CPP, name + ".cpp"),
              f"-L{libdir}", "-llbm", f"-L{LIBDIR}", "-llbm_hip",
              f"-Wl,-rpath,{libdir}:{LIBDIR}", "-o", out + ".tmp"])
        os.replace(out + ".tmp", out)
        return out

    with cf.ThreadPoolExecutor(len(CPP_SUITES)) as ex:
        return [lib] + list(ex.map(one, CPP_SUITES))


def build_all() -> list[str]:
    if shutil.which(HIPCC) is None and not os.path.exists(HIPCC):
        raise RuntimeError(f"hipcc not found at {HIPCC}")
    out = [build_hip(), build_facade()]
    out += build_cpp_suites()
    out.append(build_cli())
    return out


if __name__ == "__main__":
    for p in (build_sanitized() if "--sanitize" in sys.argv[1:] else build_all()):
        print(p)
