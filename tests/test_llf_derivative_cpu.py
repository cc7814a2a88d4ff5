"""The LLF flux's tangent and adjoint against the forward function the kernels run
(flux_llf in physics.hpp).  Bounds as for the other pointwise derivatives
(test_ad_pointwise_cpu.py): central differences of step 1e-7 leave the rounding of
the flux over the step, a few 1e-9 to 1e-8 of a derivative, and the dot products some
tens of roundings."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_llf_derivatives_of_the_kernels_flux(tmp_path):
    exe = tmp_path / "llf_check"
    subprocess.run(["g++", "-std=c++20", "-O2", "-ffp-contract=off", "-o", str(exe),
                    os.path.join(HERE, "native", "llf_check.cpp")], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    w = r.stdout.split()
    print(r.stdout)
    assert float(w[1]) <= 1e-6 and float(w[3]) <= 1e-13, r.stdout
