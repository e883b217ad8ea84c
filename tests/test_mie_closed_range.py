"""Which spheres the closed form of the Mie coefficients takes
(csrc/mie_device.h), built for the host from the same source: the downward
recurrences of every sphere it accepts stay in the range of a double, over
indices far below one as well.  CPU only: hipcc builds the host side.
"""
import cmath
import math
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "bimsim-cuda_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

DRIVER = r"""
#include "mie_device.h"
#include <cstdio>
int main() {
    using namespace bimsim;
    double x, nr, ni;
    int Nl;
    while (std::scanf("%la %la %la %d", &x, &nr, &ni, &Nl) == 4) {
        SphereDev S{};
        S.a = x;
        S.n[0] = nr;
        S.n[1] = ni;
        S.Nl = Nl;
        const mie::MieSph m = mie::mie_sph(S, 1.0);
        const double az = std::sqrt(m.zr * m.zr + m.zi * m.zi);
        std::printf("%d %d %d\n", mie::mie_closed_form(m) ? 1 : 0, mie::mie_start_order(Nl, m.x),
                    mie::mie_start_order(Nl, az));
    }
    return 0;
}
"""


def order(x):
    return int(math.ceil(x + 4.05 * x ** (1.0 / 3.0) + 2.0))


def recurrence(z, top, n):
    """The largest magnitude of the recurrence, those of the orders n .. 0 that
    are kept, and its last two values (orders 0 and 1)."""
    f, g, c = 1e-100 + 0j, 0j, 2.0 * top + 3.0
    big, kept = 0.0, []
    for k in range(top, -1, -1):
        f, g = c / z * f - g, f
        c -= 2.0
        big = max(big, abs(f))
        if not math.isfinite(big):
            break
        if k <= n:
            kept.append(abs(f))
    return big, kept, f, g


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not found")
def test_recurrences_of_the_spheres_taken_stay_in_range(tmp_path):
    src = tmp_path / "drv.cpp"
    src.write_text(DRIVER)
    exe = tmp_path / "drv"
    r = subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-O2", "-std=c++17",
                        "-ffp-contract=off", "-I", CSRC, str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    rows = []
    for x in (0.011, 0.1, 1.0, 8.0, 40.0, 64.0, 100.0, 157.0, 160.0, 240.0, 360.0, 400.0, 777.0,
              800.0, 1655.0, 1700.0, 4000.0):
        for n in (0.01, 0.1, 0.3, 0.5, 0.8, 1.0, 1.5, 0.01 + 0.01j, 0.05 + 0.2j, 1.2 + 0.02j, 1e-3 + 0.9j):
            for extra in (0, 17):
                rows.append((x, complex(n), order(x) + extra))
    text = "".join(f"{float(x).hex()} {n.real.hex()} {n.imag.hex()} {nl}\n" for x, n, nl in rows)
    out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True).stdout
    taken = 0
    for (x, n, nl), line in zip(rows, out.strip().split("\n")):
        closed, top_x, top_z = (int(v) for v in line.split())
        if not closed:
            continue
        taken += 1
        z = n * x
        for arg, top in ((complex(x), top_x), (z, top_z)):
            big, kept, f, g = recurrence(arg, top, nl)
            assert big < 1e250, (x, n, nl)
            # scaled to the larger of j_0 and j_1 no order kept is subnormal
            j0 = cmath.sin(arg) / arg
            j1 = (j0 - cmath.cos(arg)) / arg
            s = j0 / f if abs(j0) > abs(j1) else j1 / g
            assert min(kept) * abs(s) > 1e-290, (x, n, nl)
    assert taken > 100
