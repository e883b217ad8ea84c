// Device side of the FP64 Mie coefficients (sphere::calcCoeff, reference
// sphere.cpp:21-97): the three Bessel parts of a block of spheres, one wave
// each, and the coefficient formula per (sphere, order).  Shared by the
// coefficient kernels and the batch's fused pre-pass launch; every file
// that includes it is built with -ffp-contract=off.
//
// Two forms.  The general one runs the reference's CJYVA (power series or
// asymptotic expansions for the start values, start orders by its secant
// search), for any order and argument.  The closed form below it covers the
// spheres whose order belongs to their size (mie_closed_form): at half-odd
// orders the start values are sin z / z and cos z / z, so a sphere is three
// short recurrences and one quotient per order.  Both are bound by the
// latency of one sphere's chain, not by throughput; the general form's was
// mostly instruction fetch of its long straight-line code.
#pragma once

#include <algorithm>

#include "internal.h"
#include "zj_device.h"

namespace bimsim {
namespace mie {

using zj::zc;

constexpr int kSphPerLaunch = 32;   // spheres per block at most
constexpr size_t kMieLds = 61440;   // LDS budget of a block's Bessel arrays (plus 2 KB static)

constexpr int kLanes = 3;            // parts per sphere: one wave each
constexpr int kWave = 64;
constexpr int kMieThreads = (kLanes + 1) * kWave;   // and a wave for the start orders
static_assert(kSphPerLaunch <= kWave, "one lane per sphere in each part's wave");

// Spheres per block so that 2 sets x 4 arrays x wstride complex values
// per sphere fit the LDS budget.
inline int mie_spheres_per_block(int wstride) {
    const size_t per = 2 * 4 * sizeof(zc) * (size_t)wstride;
    return (int)std::max<size_t>(1, std::min<size_t>(kSphPerLaunch, kMieLds / per));
}

// The argument of part `role` of sphere S: ka for J and Y of ka (roles 0,
// 1), kna for J of kna (role 2).
__device__ inline zc mie_arg(const SphereDev& S, double kmag, int role) {
    const zc nc = {S.n[0], S.n[1]};
    return role < 2 ? zc{kmag * S.a, 0.0} : zj::zsc(S.a, zj::zsc(kmag, nc));
}

// A_l and B_l of sphere S from its two Bessel sets (w: ka set, then kna).
__device__ inline void mie_order(const SphereDev& S, int l, const zc* w, int wstride, double2* A,
                          double2* B) {
    const zc *j1 = w, *y1 = w + wstride, *jp1 = w + 2 * wstride, *yp1 = w + 3 * wstride;
    const zc *j2 = w + 4 * wstride, *jp2 = w + 6 * wstride;
    const zc nc = {S.n[0], S.n[1]};
    const zc ci = {0.0, 1.0};
    // i^l by exact repeated squaring, as std::pow(complex, int)
    const zc ipow[4] = {{1.0, 0.0}, {0.0, 1.0}, {-1.0, 0.0}, {-0.0, -1.0}};
    const zc h = zj::zadd(j1[l], zj::zmul(ci, y1[l]));
    const zc hp = zj::zadd(jp1[l], zj::zmul(ci, yp1[l]));
    const zc num_a = zj::zsub(zj::zmul(j1[l], hp), zj::zmul(jp1[l], h));
    const zc den = zj::zsub(zj::zmul(j2[l], hp), zj::zmul(zj::zmul(h, jp2[l]), nc));
    const zc f = zj::zsc(2.0 * l + 1.0, ipow[l & 3]);
    const zc An = zj::zmul(f, zj::zdiv(num_a, den));
    const zc num_b = zj::zsub(zj::zmul(zj::zmul(j1[l], jp2[l]), nc), zj::zmul(j2[l], jp1[l]));
    const zc Bn = zj::zmul(f, zj::zdiv(num_b, den));
    A[S.coeff_off + l] = make_double2(An.r, An.i);
    B[S.coeff_off + l] = make_double2(Bn.r, Bn.i);
}

// Coefficients of the block's cnt spheres (sh, wavenumbers kh, in LDS);
// lds holds 8 wstride complex values per sphere (j, y, j', y' of ka, then
// of kna).  Wave r < 3 computes part r of sphere (lane): J of ka, Y of ka,
// J of kna, as sph_jy_cplx (cbessjyva_sph) with the array clearing left out
// (every order up to Nl is written on every path).  The start orders of the
// Miller recurrences depend only on |z| and Nl, so wave 3 computes them, one
// secant search per lane, while waves 0-2 evaluate the start values; the
// parts then finish with them.  Every thread of the block (at least
// kMieThreads) then takes (sphere, order) pairs of the coefficient formula.
__device__ __forceinline__ void mie_block(const SphereDev* sh, const double* kh, int cnt,
                                          int quirks, zc* lds, int wstride, double2* A,
                                          double2* B) {
    __shared__ zj::CjyvaOrders ord[kSphPerLaunch][2];   // (sphere, ka / kna)
    const int t = (int)threadIdx.x;
    const int s = t % kWave, role = t / kWave;
    const bool part = s < cnt && role < kLanes;
    zc z = {0.0, 0.0};
    zc* o = lds;
    bool want_y = false, want_j = false;
    zj::CjyvaStart st = {};
    if (part) {
        z = mie_arg(sh[s], kh[s], role);
        o = lds + (size_t)8 * s * wstride + (role < 2 ? 0 : 4 * wstride);
        want_y = role == 1;
        want_j = role != 1 || z.i != 0.0;
        st = zj::cjyva_start(sh[s].Nl + 0.5, z, o, o + wstride, o + 2 * wstride, o + 3 * wstride,
                             quirks != 0, want_y, want_j);
    } else if (role == kLanes) {
        // one search per lane: (sphere, argument, m1 or m2)
        for (int q = s; q < 4 * cnt; q += kWave) {
            const int i = q >> 2, arg = (q >> 1) & 1, which = q & 1;
            const double v = sh[i].Nl + 0.5;
            const int m = zj::cjyva_order(zj::zabs(mie_arg(sh[i], kh[i], 2 * arg)), (int)v, which);
            if (which)
                ord[i][arg].m2 = m;
            else
                ord[i][arg].m1 = m;
        }
    }
    __syncthreads();
    if (part) {
        if (!st.done)
            zj::cjyva_rest(st, z, &ord[s][role < 2 ? 0 : 1], o, o + wstride, o + 2 * wstride,
                           o + 3 * wstride, want_y, want_j);
        zj::sph_jy_scale(sh[s].Nl, z, quirks != 0, o, o + wstride, o + 2 * wstride,
                         o + 3 * wstride, want_y, want_j);
    }
    __syncthreads();
    int lm = 0;
    for (int i = 0; i < cnt; ++i) lm = max(lm, sh[i].Nl);
    const int per = lm + 1;
    for (int idx = t; idx < cnt * per; idx += (int)blockDim.x) {
        const int i = idx / per, l = idx - i * per;
        if (l <= sh[i].Nl) mie_order(sh[i], l, lds + (size_t)8 * i * wstride, wstride, A, B);
    }
}

// ---------------------------------------------------------- closed form
// Spheres per block: few, so that the quotients (one per order) spread over
// the chip as well.
constexpr int kClosedSph = 8;
constexpr int kClosedThreads = 256;

// One sphere's input to the coefficients.
struct MieSph {
    double x, zr, zi;   // k a and n k a
    double nr, ni;
    int Nl, coeff_off;
};

__host__ __device__ inline MieSph mie_sph(const SphereDev& S, double kmag) {
    const zc z = zj::zsc(S.a, zj::zsc(kmag, zc{S.n[0], S.n[1]}));
    return MieSph{kmag * S.a, z.r, z.i, S.n[0], S.n[1], S.Nl, S.coeff_off};
}

// First order of the downward recurrence for orders up to n of argument
// magnitude az: far enough past both that what the start leaves out of
// order n (the ratio of j to y at the start against that at n, which falls
// as exp(-(2 sqrt(2)/3) 2 (d/az^(1/3))^(3/2)) past the turning point, d
// orders beyond it) is below 1e-18.
__host__ __device__ inline int mie_start_order(int n, double az) {
    const double c = cbrt(az);
    return (int)(fmax((double)n, az) + 8.0 * c + 16.0);
}

// Natural log of the growth of that recurrence from its start down to the
// orders of az's own size: v acosh(v / az) - sqrt(v^2 - az^2), v = k + 1/2
// (the ratio of j there to j at the start by their Debye expansions).  An
// absorbing sphere's grows by up to |Im z| more.
inline double mie_growth(int n, double az) {
    const double v = std::max(mie_start_order(n, az) + 0.5, az);
    return v * std::acosh(v / az) - std::sqrt(v * v - az * az);
}

// The spheres the closed form takes: the order within 20 of the size's own
// (sphere::calcNl: x + 4 x^(1/3) + 2), arguments whose sinh and cosh stay far
// from overflow, and recurrences that grow by at most exp(500) = 1e217 from
// their start of 1e-100, so that neither they nor the scaled j_l leave the
// range of a double.  Of those orders k a's grows by exp(300) at most, and so
// does an n k a no smaller; the last condition shuts out orders far beyond
// |n| k a (at n = 0.1 from k a of about 155 on, at n = 0.5 of 770).
inline bool mie_closed_form(const MieSph& m) {
    const double az = std::sqrt(m.zr * m.zr + m.zi * m.zi);
    return m.Nl >= 2 && m.x >= 1e-2 && m.x <= 4096.0 && az >= 1e-2 && az <= 4096.0 &&
           m.zr >= 0.0 && std::fabs(m.zi) <= 100.0 &&
           (double)m.Nl <= m.x + 4.05 * std::cbrt(m.x) + 20.0 &&
           (az >= m.x || mie_growth(m.Nl, az) + std::fabs(m.zi) <= 500.0);
}

// LDS of a sphere in doubles: orders 0 .. Nl of j (of ka, unscaled), y (of
// ka), j (of n ka, complex, unscaled), w = lmax + 2 each, and the scales.
__host__ __device__ inline int mie_closed_doubles(int w) { return 4 * w + 4; }

// Spherical j_0 and j_1 of z, u = 1/z.
__host__ __device__ __forceinline__ void sph_j01(double zr, double zi, double ur, double ui, zc* j0,
                                                 zc* j1) {
    double sr, cr;
    sincos(zr, &sr, &cr);
    const double e = exp(zi), ei = 1.0 / e;
    const double ch = 0.5 * (e + ei);
    // sinh near zero by its series (the difference would cancel); what it
    // leaves out is zi^12 / 13!, 1e-17 at a quarter
    const double q = zi * zi;
    const double sh_s =
        zi * (1.0 + q * (1.0 / 6.0 +
                         q * (1.0 / 120.0 +
                              q * (1.0 / 5040.0 + q * (1.0 / 362880.0 + q * (1.0 / 39916800.0))))));
    const double shi = fabs(zi) < 0.25 ? sh_s : 0.5 * (e - ei);
    const zc u = {ur, ui};
    *j0 = zj::zmul(zc{sr * ch, cr * shi}, u);
    *j1 = zj::zsub(zj::zmul(*j0, u), zj::zmul(zc{cr * ch, -(sr * shi)}, u));
}

// Coefficients of cnt <= kClosedSph spheres sh (in LDS); lds as above per
// sphere.  Waves 0, 1 and 2 run a part each (j of ka, y of ka, j of n ka;
// lane s: sphere s), then the block's threads take the (sphere, order)
// quotients.
__device__ __forceinline__ void mie_closed_block(const MieSph* sh, int cnt, int quirks, double* lds,
                                                 int w, double2* A, double2* B) {
    const int t = (int)threadIdx.x;
    const int s = t % kWave, role = t / kWave;
    const int per = mie_closed_doubles(w);
    if (s < cnt && role < 3) {
        const MieSph m = sh[s];
        const int n = m.Nl;
        double* const o = lds + s * per;
        if (role == 2) {
            // j_k = (2k + 3)/z j_{k+1} - j_{k+2}, scaled to the larger of
            // sin z / z and (sin z / z - cos z) / z at the end
            const double az2 = m.zr * m.zr + m.zi * m.zi, inv = 1.0 / az2;
            const double ur = m.zr * inv, ui = -(m.zi * inv);
            zc j0, j1;
            sph_j01(m.zr, m.zi, ur, ui, &j0, &j1);
            double fr = 1e-100, fi = 0.0, gr = 0.0, gi = 0.0;   // orders k + 1 and k + 2
            const int top = mie_start_order(n, sqrt(az2));
            double c = 2.0 * top + 3.0;
#pragma clang loop unroll_count(2)
            for (int k = top; k >= 0; --k) {
                const double ar = c * ur, ai = c * ui;
                const double hr = fma(ar, fr, fma(-ai, fi, -gr));
                const double hi = fma(ar, fi, fma(ai, fr, -gi));
                if (k <= n) {
                    o[2 * w + 2 * k] = hr;
                    o[2 * w + 2 * k + 1] = hi;
                }
                gr = fr;
                gi = fi;
                fr = hr;
                fi = hi;
                c -= 2.0;
            }
            const bool use0 = j0.r * j0.r + j0.i * j0.i > j1.r * j1.r + j1.i * j1.i;
            const zc sc = use0 ? zj::zdiv(j0, zc{fr, fi}) : zj::zdiv(j1, zc{gr, gi});
            o[4 * w + 1] = sc.r;
            o[4 * w + 2] = sc.i;
        } else {
            const double inv = 1.0 / m.x;
            double sn, cs;
            sincos(m.x, &sn, &cs);
            if (role == 0) {
                const double j0 = sn * inv, j1 = fma(j0, inv, -(cs * inv));
                double f = 1e-100, g = 0.0;
                const int top = mie_start_order(n, m.x);
                double c = 2.0 * top + 3.0;
#pragma clang loop unroll_count(2)
                for (int k = top; k >= 0; --k) {
                    const double h = fma(c * inv, f, -g);
                    if (k <= n) o[k] = h;
                    g = f;
                    f = h;
                    c -= 2.0;
                }
                o[4 * w] = fabs(j0) > fabs(j1) ? j0 / f : j1 / g;
            } else {
                // y_0 above 12: with quirks the reference's expansion adds
                // cos(x - pi/2) = sin x (its q is zero at this order)
                const double yt = -(cs * inv);
                double g = quirks && m.x > 12.0 ? (sn - cs) * inv : yt;
                double f = fma(yt, inv, -(sn * inv));
                o[w] = g;
                o[w + 1] = f;
                double c = 3.0;
#pragma clang loop unroll_count(2)
                for (int k = 2; k <= n; ++k) {
                    const double h = fma(c * inv, f, -g);
                    o[w + k] = h;
                    g = f;
                    f = h;
                    c += 2.0;
                }
            }
        }
    }
    __syncthreads();
    int lm = 0;
    for (int i = 0; i < cnt; ++i) lm = max(lm, sh[i].Nl);
    const int nl = lm + 1;
    for (int idx = t; idx < cnt * nl; idx += (int)blockDim.x) {
        const int i = idx / nl, l = idx - i * nl;
        const MieSph& m = sh[i];
        if (l > m.Nl) continue;
        const double* const o = lds + i * per;
        const double* const Y = o + w;
        const double* const K = o + 2 * w;
        const double js = o[4 * w], ix = 1.0 / m.x;
        const zc ks = {o[4 * w + 1], o[4 * w + 2]};
        // the derivatives f_l' = f_{l-1} - (l + 1)/z f_l (f_0' = -f_1)
        const int lo = l > 0 ? l - 1 : 1;
        const double sg = l > 0 ? 1.0 : -1.0, c = l > 0 ? l + 1.0 : 0.0;
        const double j1 = o[l] * js, y1 = Y[l];
        const double jp1 = fma(-(c * ix), j1, sg * (o[lo] * js));
        const double yp1 = fma(-(c * ix), y1, sg * Y[lo]);
        const zc j2 = zj::zmul(zc{K[2 * l], K[2 * l + 1]}, ks);
        const zc jl = zj::zmul(zc{K[2 * lo], K[2 * lo + 1]}, ks);
        const zc jp2 = zj::zsub(zj::zsc(sg, jl), zj::zmul(zj::rdiv(c, zc{m.zr, m.zi}), j2));
        const zc nc = {m.nr, m.ni};
        const zc h = {j1, y1}, hp = {jp1, yp1};
        const zc den = zj::zsub(zj::zmul(j2, hp), zj::zmul(zj::zmul(h, jp2), nc));
        // j1 h' - j1' h = i (j1 y1' - j1' y1)
        const zc num_a = {0.0, fma(j1, yp1, -(jp1 * y1))};
        const zc num_b = zj::zsub(zj::zmul(zj::zsc(j1, jp2), nc), zj::zsc(jp1, j2));
        const double f = 2.0 * l + 1.0;
        const zc il = {(l & 1) ? 0.0 : ((l & 2) ? -f : f), (l & 1) ? ((l & 2) ? -f : f) : 0.0};
        const zc An = zj::zmul(il, zj::zdiv(num_a, den));
        const zc Bn = zj::zmul(il, zj::zdiv(num_b, den));
        A[m.coeff_off + l] = make_double2(An.r, An.i);
        B[m.coeff_off + l] = make_double2(Bn.r, Bn.i);
    }
}

}  // namespace mie
}  // namespace bimsim
