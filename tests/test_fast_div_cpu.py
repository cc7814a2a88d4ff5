"""The multiply-high division the kernels take element indices apart with
(FastDiv in kernels.hpp) equals the integer division over its whole range."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_fast_div_equals_division(tmp_path):
    exe = tmp_path / "fast_div"
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-std=c++20", "-O2", "-D__HIP_PLATFORM_AMD__", f"-I{rocm}/include", "-o", str(exe),
                    os.path.join(HERE, "native", "fast_div.cpp")], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.startswith("ok "), r.stdout
