"""The order of a slice's pixels by the sphere that holds them, as the harmonic
plan's host code finds it (chords of the rows), against the test of every pixel
and sphere: rotated, skewed, tilted, mirrored and stretched slices, spheres on
their edges, smaller than a pixel, larger than the slice, overlapping, far
away.  CPU only: a host program on the built library.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "bimsim-cuda_amd")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

DRIVER = r"""
#include "us_series.h"
#include <cstdio>
#include <cstring>
#include <random>
using namespace bimsim;
int main() {
    std::mt19937_64 g(7);
    auto U = [&](double lo, double hi) { return std::uniform_real_distribution<double>(lo, hi)(g); };
    long long held = 0, wrong = 0;
    for (int k = 0; k < 600; ++k) {
        bool some = false;
        SeriesInst I;
        std::memset(&I, 0, sizeof I);
        I.uR = 1 + (int)(g() % 90);
        I.vR = 1 + (int)(g() % 90);
        I.ns = (int)(g() % 6);
        const double L = k % 7 == 0 ? 1e-3 : 40.0, at = k % 11 == 0 ? 1e5 : 0.0;
        auto edge = [&](int c) {
            return d3{c == 0 ? U(-L, L) : k % 3 ? 0.0 : U(-L, L), c == 1 ? U(-L, L) : k % 3 ? 0.0 : U(-L, L),
                      k % 5 ? 0.0 : U(-L, L)};
        };
        I.q.X = edge(0);
        I.q.Y = edge(1);
        if (k % 50 == 0) I.q.X = d3{0.0, 0.0, 0.0};
        I.q.A = d3{at + U(-L, L), at + U(-L, L), k % 5 ? 0.0 : U(-L, L)};
        std::vector<SeriesSph> sph(I.ns);
        for (SeriesSph& S : sph) {
            std::memset(&S, 0, sizeof S);
            // a centre on a pixel or anywhere about the slice
            const d3 p = g() % 2 ? quad_at(I.q, (double)(g() % I.uR) / I.uR, (double)(g() % I.vR) / I.vR)
                                 : quad_at(I.q, U(-0.5, 1.5), U(-0.5, 1.5));
            S.s.p[0] = p.x;
            S.s.p[1] = p.y;
            S.s.p[2] = p.z + (g() % 3 ? 0.0 : U(-0.2, 0.2) * L);
            S.s.a = L * (g() % 4 == 0 ? 1e-4 : g() % 4 == 0 ? 3.0 : U(0.01, 0.4));
            // a radius that ends exactly on a pixel
            if (g() % 4 == 0)
                S.s.a = len(sub(quad_at(I.q, (double)(g() % I.uR) / I.uR, (double)(g() % I.vR) / I.vR),
                                mk(S.s.p))) + 1e-300;
        }
        std::vector<int> cls(I.uR * I.vR, 0), perm(3, -1), want(3, -1);
        for (int pix = 0; pix < I.uR * I.vR; ++pix) {
            const int iv = pix / I.uR, iu = pix - iv * I.uR;
            const d3 p = quad_at(I.q, (double)iu / (double)I.uR, (double)iv / (double)I.vR);
            for (int t = 0; t < I.ns && !cls[pix]; ++t)
                if (len(sub(p, mk(sph[t].s.p))) <= sph[t].s.a) cls[pix] = t + 1;
            held += cls[pix] > 0;
            some = some || cls[pix] > 0;
        }
        // by class, the pixels of none last, each class as it comes
        for (int c = 1; some && c <= I.ns + 1; ++c)
            for (int pix = 0; pix < I.uR * I.vR; ++pix)
                if (cls[pix] == c % (I.ns + 1)) want.push_back(pix);
        wrong += pixel_order(I, sph.data(), &perm) != some || perm != want;
    }
    std::printf("%lld %lld\n", held, wrong);
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC) or
                    not os.path.exists(os.path.join(PKG, "libbimsim_hip.so")),
                    reason="needs hipcc and a build")
def test_chords_give_the_same_order(tmp_path):
    src, exe = tmp_path / "drv.cpp", tmp_path / "drv"
    src.write_text(DRIVER)
    r = subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-O2", "-std=c++17",
                        "-ffp-contract=off", "-I", os.path.join(PKG, "csrc"), str(src), "-o",
                        str(exe), "-L", PKG, "-lbimsim_hip", f"-Wl,-rpath,{PKG}"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    held, wrong = (int(v) for v in out.split())
    assert held > 10000 and wrong == 0
