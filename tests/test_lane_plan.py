"""Host code of the wave kernels, compiled without device code."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _run(tmp_path, name):
    exe = str(tmp_path / name)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-D__HIP_PLATFORM_AMD__", "-isystem",
                    "/opt/rocm/include", "-I",
                    os.path.join(ROOT, "spinparser_amd", "csrc"), "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", name + ".cpp")], check=True, timeout=300)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0 and res.stdout == "ok\n", res.stdout + res.stderr


def test_overlap_plan(tmp_path):
    """Lanes' sums equal the lists', in both storages; the fixed one allocates nothing."""
    _run(tmp_path, "lane_plan_test")


def test_buffers_of_the_atomics(tmp_path):
    """Only ordinary memory of the device that runs the kernel is added to with atomics."""
    _run(tmp_path, "atomic_memory_test")
