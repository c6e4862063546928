"""How work is cut into workgroups (csrc/densify_grid.h, csrc/deal.h): the host arithmetic, compiled and run on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_dispatch_arithmetic(tmp_path):
    exe = tmp_path / "dispatch_check"
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"), "-I", os.path.join(ROOT, "deploy3d_amd", "csrc"),
                           os.path.join(ROOT, "tests", "dispatch_host", "dispatch_check.cpp"), "-o", str(exe)])
    res = subprocess.run([str(exe)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert res.returncode == 0 and "dispatch_check ok" in res.stdout, res.stdout
