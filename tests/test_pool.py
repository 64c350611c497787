"""The pool of tensors' device memory, compiled against a HIP that only counts (tests/cpp/pool_test.cpp): no GPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_pool_against_a_counting_hip(tmp_path):
    exe = str(tmp_path / "pool_test")
    cc = subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-isystem", "/opt/rocm/include",
                         os.path.join(ROOT, "tests", "cpp", "pool_test.cpp"), "-o", exe, "-lpthread"], capture_output=True, text=True)
    assert cc.returncode == 0, cc.stderr[-3000:]
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and run.stdout.strip() == "OK", run.stdout + run.stderr
