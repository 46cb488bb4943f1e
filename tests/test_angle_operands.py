"""The key of the angular operator's cached operands, built for the host alone:
calls that take different kernels, or differ in any table or size the operands
are made from, never share them."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

MAIN = r"""
#include "angle_operands.hpp"
#include <cstdio>
using namespace bfpn;
int main() {
    const double sig[500] = {1.0, 2.0}, other[500] = {1.0, 3.0};
    // 500 groups of 20 x 20 directions: 2^31 values between 10,737 and 10,738 nodes
    auto matrix = [](int nyz, int n, int Ng) {
        return angle_on_matrix_cores(n, n, static_cast<long long>(Ng) * nyz);
    };
    auto key = [&](bool fp64, int nyz, int Nmu = 20, int Nom = 20, double du = 0.1, double dv = 0.2,
                   double dt = 0.02, double rho = 1.0, const double* s = nullptr, int Ng = 500) {
        const bool m = !fp64 && angle_on_matrix_cores(Nmu, Nom, static_cast<long long>(Ng) * nyz);
        return angle_operand_key(fp64, m, Ng, Nmu, Nom, du, dv, dt, rho, s ? s : sig);
    };
    int bad = 0;
    auto check = [&](bool ok, const char* what) {
        if (!ok) std::printf("%s\n", what), ++bad;
    };
    check(matrix(10737, 20, 500) && !matrix(10738, 20, 500), "limit in values");
    check(matrix((1 << 30) - 1, 1, 1) && !matrix(1 << 30, 1, 1), "limit in planes");
    check(!matrix(1, 33, 1), "widest plane");
    const auto k = key(false, 441);
    check(k == key(false, 10737), "same kernel, other nodes");
    check(k != key(false, 10738), "other kernel");
    check(key(false, 10738) == key(false, 20000), "same vector kernel");
    check(k != key(true, 441), "precision");
    check(key(true, 441) == key(true, 10738), "one FP64 kernel");
    check(key(false, 441, 20, 16) != key(false, 441, 16, 20), "sizes in order");
    check(k != key(false, 441, 20, 20, 0.2), "du");
    check(k != key(false, 441, 20, 20, 0.1, 0.1), "dv");
    check(k != key(false, 441, 20, 20, 0.1, 0.2, 0.01), "dt");
    check(k != key(false, 441, 20, 20, 0.1, 0.2, 0.02, 2.0), "density");
    check(k != key(false, 441, 20, 20, 0.1, 0.2, 0.02, 1.0, other), "table");
    check(k != key(false, 441, 20, 20, 0.1, 0.2, 0.02, 1.0, sig, 400), "groups");
    return bad;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_operand_key(tmp_path):
    src, exe = tmp_path / "key.cpp", tmp_path / "key"
    src.write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", f"-I{os.path.join(ROOT, 'bfpn_gpu_amd', 'csrc')}", "-o",
                    str(exe), str(src)], check=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=30)
    assert r.returncode == 0, r.stdout
