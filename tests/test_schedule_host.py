"""The schedule's host code (csrc/schedule.cpp, csrc/schedule_capture.cpp) against a stand-in for the HIP runtime: when graphs are
captured, dropped and destroyed, what a captured pass is made of, and that none of it waits for the device or spoils a capture of
the caller's.  Compiled and run on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_schedule_host_code(tmp_path):
    exe = tmp_path / "schedule_check"
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"),
                           "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "deploy3d_amd", "csrc"),
                           os.path.join(ROOT, "deploy3d_amd", "csrc", "schedule.cpp"),
                           os.path.join(ROOT, "deploy3d_amd", "csrc", "schedule_capture.cpp"),
                           os.path.join(ROOT, "tests", "schedule_host", "schedule_check.cpp"), "-o", str(exe)])
    res = subprocess.run([str(exe)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert res.returncode == 0 and "schedule_check ok" in res.stdout, res.stdout
