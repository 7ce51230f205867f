"""The pinned slots of the host copies (lbm_transfer.hip) on a stand-in for
the HIP runtime: tests/cpp/TransferPool.cpp, built here by g++ together with
the file itself."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_slots_are_kept_shared_and_given_back(tmp_path):
    exe = str(tmp_path / "TransferPool")
    source = os.path.join(ROOT, "latticeboltzmanncuda_amd", "csrc",
                          "lbm_transfer.hip")
    r = subprocess.run(
        ["g++", "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__",
         "-I/opt/rocm/include", "-I" + os.path.join(ROOT, "include"),
         os.path.join(ROOT, "tests", "cpp", "TransferPool.cpp"),
         "-x", "c++", source, "-o", exe,
         "-L/opt/rocm/lib", "-lrocprofiler-sdk-roctx",
         "-Wl,-rpath,/opt/rocm/lib"],
        capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr
