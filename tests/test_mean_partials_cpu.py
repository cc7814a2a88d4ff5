"""The partial derivatives of the two-point flux's means (physics_ad.hpp)
against long double, over every branch and its edges.  Bound, in double
epsilons of the mean over its argument: a partial takes about 30 roundings of
half an epsilon (a reciprocal, the ratio, two series, and their products)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_mean_partials_against_long_double(tmp_path):
    exe = tmp_path / "mean_partials"
    subprocess.run(["g++", "-std=c++20", "-O2", "-ffp-contract=off", "-o", str(exe),
                    os.path.join(HERE, "native", "mean_partials.cpp")], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
    assert float(r.stdout.split()[1]) <= 15.0, r.stdout
