"""The operators' host code (csrc/plugin.cpp) against stand-ins for the HIP runtime and the kernels: what an enqueue reserves,
where and for how long, and which layers sort the rows of their table.  Compiled and run on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_plugin_host_code(tmp_path):
    exe = tmp_path / "plugin_check"
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"),
                           "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "deploy3d_amd", "csrc"),
                           os.path.join(ROOT, "deploy3d_amd", "csrc", "plugin.cpp"),
                           os.path.join(ROOT, "tests", "plugin_host", "plugin_check.cpp"), "-ldl", "-o", str(exe)])
    env = {k: v for k, v in os.environ.items() if k != "D3D_DEBUG_ENV"}
    res = subprocess.run([str(exe)], env=env, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert res.returncode == 0 and "plugin_check ok" in res.stdout, res.stdout
