"""mmp_fiber_load that fails half-way (tests/cpp/load_failures.cpp): every copy and synchronisation of a load that
changes the batch's plan fails once, in a program that stands in for the HIP runtime. No device is needed."""
import os
import shutil
import subprocess

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CPP = os.path.join(REPO, "tests", "cpp")
LIB = os.path.join(REPO, "mm_propagation_amd", "lib")


def test_load_failures(tmp_path):
    exe = str(tmp_path / "load_failures")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    r = subprocess.run([shutil.which("g++") or "g++", "-std=c++17", "-O1", "-Wall", "-D__HIP_PLATFORM_AMD__", "-rdynamic",
                        "-isystem", rocm + "/include", "-I" + os.path.join(REPO, "include"), os.path.join(CPP, "load_failures.cpp"),
                        "-o", exe, "-L" + LIB, "-lmmprop_hip", "-Wl,-rpath," + LIB, "-Wl,--allow-shlib-undefined"],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "load failure checks passed" in r.stdout, r.stdout[-1000:] + r.stderr[-4000:]
