"""The normal deviates of a network's initial weights (sf_normal.h) are the sequence of
std::normal_distribution<double> on the same generator, so that a seed gives the same network: both
are compiled here from the header and compared, deviate for deviate."""
import os
import shutil
import subprocess

import pytest

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "starfish_amd", "csrc", "sf_normal.h")
SOURCE = r"""
#include <cstdio>
#include "%s"
int main() {
    const double sigma[] = {1.0, 0.2357022603955158, 0.08838834764831845, 1e-3};
    for (unsigned long long seed : {0ull, 1ull, 3ull, 2024ull, 0x9E3779B97F4A7C15ull}) {
        std::mt19937_64 ra(seed), rb(seed);
        for (double s : sigma) {
            sf::PolarNormal a{s};
            std::normal_distribution<double> b(0.0, s);
            for (int k = 0; k < 100001; k++) {   // (an odd count: the kept deviate goes with the object)
                const double x = a(ra), y = b(rb);
                if (!(x == y)) return std::printf("seed %%llu sigma %%g draw %%d: %%.17g, not %%.17g\n", seed, s, k, x, y), 1;
            }
            if (ra != rb) return std::printf("the generators differ after sigma %%g\n", s), 1;
        }
    }
    return 0;
}
"""


def test_weights_are_the_standard_librarys_deviates(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    src, exe = tmp_path / "normal.cpp", tmp_path / "normal"
    src.write_text(SOURCE % HEADER)
    subprocess.run([gxx, "-O2", "-std=c++17", "-o", str(exe), str(src)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
