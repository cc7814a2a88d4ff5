"""The kernels' logarithmic means and two-point flux (physics.hpp) against long
double, over every branch and its edges.

Bounds, in double epsilons: artanh(xi)/xi takes at most a reciprocal, a
product, a series and a quotient, under 16 roundings of half an epsilon; a flux
component takes fewer than 16 more, each against the magnitudes it sums."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_pair_flux_against_long_double(tmp_path):
    exe = tmp_path / "pair_flux"
    subprocess.run(["g++", "-std=c++20", "-O2", "-ffp-contract=off", "-o", str(exe),
                    os.path.join(HERE, "native", "pair_flux.cpp")], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
    w = r.stdout.split()
    assert float(w[1]) <= 8.0 and float(w[3]) <= 16.0, r.stdout
    assert w[5] == "1" and w[7] == "1", r.stdout
