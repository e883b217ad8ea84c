"""Which plans of the harmonic form take nodes (csrc/us_nodes.h): the faster of
the two at sizes on either side of the line where both were measured, and the
calls of test_gpu_nodes.py, which are there to test the nodes.  CPU only: a
host program on the built library.
"""
import math
import os
import shutil
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "bimsim-cuda_amd")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

DRIVER = r"""
#include "us_nodes.h"
#include <cstdio>
#include <cstring>
using namespace bimsim;
int main() {
    int uR, vR, ns;
    double k, q[9];
    while (std::scanf("%d %d %d %lf", &uR, &vR, &ns, &k) == 4) {
        for (double& x : q)
            if (std::scanf("%lf", &x) != 1) return 1;
        SeriesInst I;
        std::memset(&I, 0, sizeof I);
        I.uR = uR;
        I.vR = vR;
        I.ns = ns;
        I.kmag = k;
        I.q.A = mk(q);
        I.q.X = mk(q + 3);
        I.q.Y = mk(q + 6);
        std::vector<SeriesSph> sph(ns);
        bool planar = q[5] == 0.0 && q[8] == 0.0;
        for (SeriesSph& S : sph) {
            std::memset(&S, 0, sizeof S);
            if (std::scanf("%lf %lf %lf %lf %d", S.s.p, S.s.p + 1, S.s.p + 2, &S.s.a, &S.s.Nl) != 5)
                return 1;
            planar = planar && S.s.p[2] == q[2];
        }
        NodeTables t;
        const NodeCost p = node_pixel_cost(I, sph.data(), planar);
        const NodeCost n = node_plan_instance(I, sph.data(), planar, &t);
        std::printf("%d\n", t.inst[0].n_lev > 0 && n.total() < p.total() ? t.inst[0].n_lev : 0);
    }
}
"""


@pytest.fixture(scope="module")
def levels(tmp_path_factory):
    """Tile sizes that hold nodes, for calls (A, X, Y, uR, vR, k, spheres)."""
    if not os.path.exists(HIPCC) or not os.path.exists(os.path.join(PKG, "libbimsim_hip.so")):
        pytest.skip("needs hipcc and a build")
    d = tmp_path_factory.mktemp("node_rule")
    src, exe = d / "drv.cpp", d / "drv"
    src.write_text(DRIVER)
    r = subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-O2", "-std=c++17",
                        "-ffp-contract=off", "-I", os.path.join(PKG, "csrc"), str(src), "-o",
                        str(exe), "-L", PKG, "-lbimsim_hip", f"-Wl,-rpath,{PKG}"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]

    def ask(calls):
        text = ""
        for A, X, Y, uR, vR, k, spheres in calls:
            text += f"{uR} {vR} {len(spheres)} {k!r}\n" + " ".join(repr(float(v)) for v in (*A, *X, *Y))
            for s in spheres:
                text += "\n" + " ".join(repr(float(v)) for v in (*s["p"], s["a"])) + f" {s['Nl']}"
            text += "\n"
        out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True)
        return [int(v) for v in out.stdout.split()]

    return ask


# N, spheres, k a of the first, width, height of the spheres over the slice; us a
# call by pixels and by nodes (400 waves, wavenumber 1.5)
MEASURED = [
    (256, 3, 25.0, 60.0, 0.0, 68.6, 91.3),
    (256, 6, 25.0, 60.0, 0.0, 104.7, 119.9), (256, 20, 25.0, 60.0, 0.0, 288.3, 229.5),
    (256, 6, 15.0, 60.0, 1.5, 214.4, 166.9), (256, 1, 25.0, 60.0, 1.5, 101.9, 117.7),
    (320, 3, 25.0, 60.0, 0.0, 70.6, 89.3), (320, 10, 25.0, 60.0, 0.0, 176.8, 146.3),
    (512, 2, 25.0, 60.0, 0.0, 74.2, 91.3), (512, 3, 25.0, 150.0, 0.0, 81.7, 97.9),
    (512, 3, 25.0, 60.0, 0.0, 93.8, 111.4), (512, 6, 25.0, 60.0, 0.0, 154.5, 134.6),
    (512, 6, 8.0, 150.0, 0.0, 69.1, 80.0), (512, 10, 25.0, 60.0, 0.0, 237.0, 178.6),
    (512, 6, 8.0, 60.0, 1.5, 146.5, 128.7), (768, 2, 8.0, 60.0, 0.0, 78.3, 56.6),
    (768, 6, 8.0, 60.0, 0.0, 110.5, 92.5), (1024, 1, 8.0, 60.0, 0.0, 89.1, 49.1),
    (1024, 3, 8.0, 60.0, 0.0, 109.0, 84.4), (1024, 3, 25.0, 60.0, 1.5, 736.4, 466.9),
]


def test_the_faster_of_the_two_where_both_were_measured(pkg, levels):
    calls, k = [], 1.5
    for N, ns, ka, width, z, _, _ in MEASURED:
        rng, spheres = np.random.default_rng(5), []
        for i in range(ns):
            a = ka / k / (1.0 + 0.02 * i)
            x, y = (0.0, 0.0) if i == 0 else rng.uniform(-0.5, 0.5, 2) * width
            spheres.append(dict(p=(x, y, z), a=a, Nl=pkg.sphere_order(a, 2.0 * math.pi / k)))
        calls.append(((-width / 2, -width / 2, 0.0), (width, 0.0, 0.0), (0.0, width, 0.0), N, N, k,
                      spheres))
    for (*case, pixels, nodes), lev in zip(MEASURED, levels(calls)):
        assert (lev > 0) == (nodes < pixels), (case, lev)


def test_the_gpu_tests_take_nodes(pkg, levels, monkeypatch):
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import test_gpu_nodes as T
    calls, names = [], []

    def both(pkg, ctx, q, uR, vR, lam, rows, **kw):
        spheres, _ = T.spheres_of(pkg, lam, rows + T.FAR)
        calls.append((list(q.A), list(q.X), list(q.Y), uR, vR, 2.0 * math.pi / lam, spheres))

    monkeypatch.setattr(T, "both", both)
    monkeypatch.setattr(T, "check", lambda *a, **kw: None)
    for name in dir(T):
        f = getattr(T, name)
        if not name.startswith("test_nodes"):
            continue
        sets = [{}]
        for m in getattr(f, "pytestmark", []):
            if m.name != "parametrize":
                continue
            keys = [v.strip() for v in m.args[0].split(",")]
            sets = [dict(s, **dict(zip(keys, v if len(keys) > 1 else (v,))))
                    for s in sets for v in m.args[1]]
        for s in sets:
            f(pkg, None, **s)
            names.append(s)
    got = levels(calls)
    assert len(got) > 25
    # (pixels too coarse for a tile's nodes: the other side of the rule)
    without = [n for n, lev in zip(names, got) if lev == 0]
    assert without == [dict(case="coarse"), dict(lam=2.5, uR=512, vR=130)]
