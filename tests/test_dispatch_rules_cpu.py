"""The compile-time rules that choose between kernels (static_asserts of
tests/native/dispatch_rules.hip, compiled for the host)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_dispatch_rules():
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    r = subprocess.run([hipcc, "-std=c++20", "--offload-host-only", "-fsyntax-only",
                        os.path.join(HERE, "native", "dispatch_rules.hip")],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
