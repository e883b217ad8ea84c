"""Spherical j_0 and j_1 of a complex argument (csrc/mie_device.h: what the
closed forms' recurrences are scaled to), built for the host from the same
source and compared with mpmath, on both sides of where sinh changes from its
series to its exponentials.  CPU only: hipcc builds the host side.
"""
import math
import os
import shutil
import subprocess

import pytest

mp = pytest.importorskip("mpmath")

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "bimsim-cuda_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

DRIVER = r"""
#include "mie_device.h"
#include <cstdio>
int main() {
    using namespace bimsim;
    double x, y;
    while (std::scanf("%la %la", &x, &y) == 2) {
        const mie::zc u = zj::rdiv(1.0, mie::zc{x, y});
        mie::zc j0, j1;
        mie::sph_j01(x, y, u.r, u.i, &j0, &j1);
        std::printf("%a %a %a %a\n", j0.r, j0.i, j1.r, j1.i);
    }
    return 0;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not found")
def test_j0_and_j1_against_mpmath(tmp_path):
    src = tmp_path / "drv.cpp"
    src.write_text(DRIVER)
    exe = tmp_path / "drv"
    r = subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-O2", "-std=c++17",
                        "-ffp-contract=off", "-I", CSRC, str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    # multiples of pi, where sin is small and sinh the whole of sin z, and others
    xs = [math.pi, 2 * math.pi, 25 * math.pi, 1.0, 7.3, 60.1]
    ys = [0.0, 1e-9, 1e-3, 0.05, 0.1, 0.2, 0.2499999, 0.25, 0.2500001, 0.4, 1.0, 5.0]
    z = [(x, s * y) for x in xs for y in ys for s in (1, -1)]
    out = subprocess.run([str(exe)], input="".join(f"{x.hex()} {y.hex()}\n" for x, y in z),
                         capture_output=True, text=True, check=True).stdout.strip().split("\n")
    mp.mp.prec = 160
    for (x, y), line in zip(z, out):
        got = [float.fromhex(v) for v in line.split()]
        c = mp.mpc(x, y)
        j0 = mp.sin(c) / c
        j1 = j0 / c - mp.cos(c) / c
        # a few products and quotients of rounded values (an ulp of sin, cos and
        # exp; two bits of sinh from its exponentials just past a quarter):
        # within 16 roundings of the sums of their terms' magnitudes
        s0 = (abs(mp.sin(x)) * mp.cosh(y) + abs(mp.cos(x) * mp.sinh(y))) / abs(c)
        s1 = s0 / abs(c) + (abs(mp.cos(x)) * mp.cosh(y) + abs(mp.sin(x) * mp.sinh(y))) / abs(c)
        assert abs(mp.mpc(got[0], got[1]) - j0) <= 16 * mp.mpf(2) ** -53 * s0, (x, y)
        assert abs(mp.mpc(got[2], got[3]) - j1) <= 16 * mp.mpf(2) ** -53 * s1, (x, y)
