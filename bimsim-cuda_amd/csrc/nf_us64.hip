// Scattered/internal field of spheres under Monte-Carlo plane waves
// (nearfieldStruct::scalarUs, reference nfScalarUs.cu:494-658), FP64.
//
// The reference evaluates, per pixel, sphere and wave, the full calc_Us /
// calc_Ui recurrences (optPc_gpuScalarUsp, nfScalarUs.cu:449-491).  Here the
// radial products c_l = B_l h_l(kd) or A_l j_l(knd), which no wave changes,
// are formed once per (pixel, sphere); every other operation is the
// reference's, in its order, and the file is built with -ffp-contract=off, so
// both FP64 precisions are this one kernel.  The FP32 form lives in
// us_series.hip.
#include "nf_us.h"
#include "us_series.h"
#include "refmath.h"

namespace bimsim {
namespace {

constexpr int kThreads = 256;
constexpr int kGroups = kThreads / 64;   // wavefronts that share a block's pixels
constexpr int kWaves = 8;                // plane waves a wavefront carries at a time
constexpr int kSum = 4;                  // of them summed at a time
constexpr int kPhases = 128;             // plane waves whose phases are held in LDS
constexpr int kSumBytes = kGroups * kSum * 64 * (int)sizeof(double2);
constexpr int kOrders = 112;             // orders whose c_l are held in LDS

// The constants of one Legendre step, P_l = ((2l-1) x P_{l-1} - (l-1) P_{l-2}) / l.
struct StepConst {
    double a, b, n, inv;
};

// a / n correctly rounded for an integer n, given inv = 1/n rounded: q is
// within 1.5 ulp, so the remainder, a multiple of q's last place no larger
// than 1.5 n of them, is exact; the corrected quotient differs from a/n by at
// most 1.5 ulp 2^-53 before it is rounded, while a/n is a midpoint of two
// doubles or nearer to one than 1/(2n) ulp never (n m, m odd of 54 bits, has
// more than 53 bits).  3 operations for the 10 or more of a division.
__device__ __forceinline__ double div_int(double a, double n, double inv) {
    const double q = a * inv;
    return fma(fma(-q, n, a), inv, q);
}

__device__ inline dc ld2(const double2* p, int i) {
    const double2 v = p[i];
    return dc{v.x, v.y};
}

// The radial products of calc_Us / calc_Ui (reference nfScalarUs.cu:50-95,
// 201-245) for one pixel and sphere, in order of l.
struct Radial {
    int kind;   // 0 = outside (Hankel), 1 = inside (Bessel), 2 = inside near
                // the centre, where calc_Ui returns A_0 for every wave
    double kd;
    dc knd;
    double j[2], y[2];   // or the complex j, split into these

    __device__ void locate(double d, double kmag, const SphereDev& S) {
        kd = kmag * d;
        knd = cscl(dc{S.n[0], S.n[1]}, kmag * d);
        kind = d <= S.a ? (knd.r < (double)kEpsFloat ? 2 : 1) : 0;
    }
    // j_l and y_l, l0 <= l < l1, to out[64 (l - l0)]; l0 = 0 or the last
    // call's l1.  The chains are wavefronts of their own: g = 0 j and 1 y
    // outside, 2 the complex j inside.
    __device__ void run(int g, int l0, int l1, double2* out) {
        if (kind == 0 && g == 0) {
            if (l0 == 0) ref::init_j(kd, j);
            for (int l = l0; l < l1; ++l) {
                if (l > 1) ref::shift_j(l, kd, j);
                out[64 * (l - l0)].x = l > 0 ? j[1] : j[0];
            }
        } else if (kind == 0 && g == 1) {
            if (l0 == 0) ref::init_y(kd, y);
            for (int l = l0; l < l1; ++l) {
                if (l > 1) ref::shift_y(l, kd, y);
                out[64 * (l - l0)].y = l > 0 ? y[1] : y[0];
            }
        } else if (kind == 1 && g == 2) {
            dc b[2] = {{j[0], y[0]}, {j[1], y[1]}};
            if (l0 == 0) ref::init_jc(knd, b);
            for (int l = l0; l < l1; ++l) {
                if (l > 1) ref::shift_jc(l, knd, b);
                const dc v = l > 0 ? b[1] : b[0];
                out[64 * (l - l0)] = make_double2(v.r, v.i);
            }
            j[0] = b[0].r, y[0] = b[0].i, j[1] = b[1].r, y[1] = b[1].i;
        }
    }
};

// What the wavefronts of a block share for one sphere.
struct Block {
    double2* c;         // [l - l0][pixel]
    StepConst* step;    // [l - l0]
    double2* ph;        // (scale*subA) * exp(i kmag k.c) of kPhases waves
    double* re;         // [wave][pixel] terms of the waves to be summed
    double* im;
    const double2 *A, *B;
    int Nl, cap;        // orders, orders held at a time
    int g, lane;
};

// The c_l of the orders [l0, l1) into LDS (after a barrier, and before one).
__device__ __forceinline__ void hold_orders(const Block& T, Radial& R, int l0, int l1) {
    R.run(T.g, l0, l1, T.c + T.lane);
    if (T.g == kGroups - 1)
        for (int l = l0 + T.lane; l < l1; l += 64)
            T.step[l - l0] =
                StepConst{(double)(2 * l - 1), (double)(l - 1), (double)l, 1.0 / (double)l};
    __syncthreads();
    for (int l = l0 + T.g; l < l1; l += kGroups) {
        double2& c = T.c[64 * (l - l0) + T.lane];
        dc v = {0.0, 0.0};
        if (R.kind < 2)
            v = cmul(ld2(R.kind == 0 ? T.B : T.A, l), dc{c.x, c.y});
        else if (l == 0)
            v = ld2(T.A, 0);
        c = make_double2(v.r, v.i);
    }
}

// kGroups x W waves from w0 on: wavefront g takes w0 + w kGroups + g, so that
// each kSum of a wavefront's W, taken over the wavefronts, follow each other.
// sum: the pixel's sum over the waves so far, its real part in wavefront 0
// and its imaginary part in wavefront 1.
template <int W>
__device__ __forceinline__ void wave_round(const Block& T, Radial& R, d3 r,
                                           const double* __restrict__ waves, int w0, int p0,
                                           int nk, double& sum) {
    constexpr int V = W < kSum ? W : kSum;
    double x[W], P0[W], P1[W], tr[W], ti[W];
    const bool active = w0 + T.g < nk;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        const int i = min(w0 + w * kGroups + T.g, nk - 1);
        x[w] = dot(mk(waves + 3 * i), r);
    }
    const int n = T.Nl + 1;
    for (int l0 = 0; l0 < n; l0 += T.cap) {
        const int l1 = min(l0 + T.cap, n);
        if (n > T.cap) {
            __syncthreads();
            hold_orders(T, R, l0, l1);
            __syncthreads();
        }
        if (!active) continue;
        const double2* c = T.c + T.lane;
        auto step = [&](int l, double* Pa, const double* Pb) {   // Pa = P_l of (Pa, Pb)
            const StepConst k = T.step[l - l0];
            const double2 cl = c[64 * (l - l0)];
#pragma unroll
            for (int w = 0; w < W; ++w) {
                Pa[w] = div_int(k.a * x[w] * Pb[w] - k.b * Pa[w], k.n, k.inv);
                tr[w] += cl.x * Pa[w];
                ti[w] += cl.y * Pa[w];
            }
        };
        int l = l0;
        if (l0 == 0) {
            const double2 c0 = c[0], c1 = c[64];
#pragma unroll
            for (int w = 0; w < W; ++w) {
                P0[w] = 1.0;
                P1[w] = x[w];
                tr[w] = 0.0 + c0.x;
                ti[w] = 0.0 + c0.y;
                tr[w] += c1.x * x[w];
                ti[w] += c1.y * x[w];
            }
            l = 2;
        }
        for (; l + 1 < l1; l += 2) {
            step(l, P0, P1);
            step(l + 1, P1, P0);
        }
        if (l < l1) {
            step(l, P0, P1);
#pragma unroll
            for (int w = 0; w < W; ++w) {
                const double t = P0[w];
                P0[w] = P1[w];
                P1[w] = t;
            }
        }
    }
#pragma unroll
    for (int h = 0; h < W; h += V) {
        __syncthreads();   // the previous sum is done
        if (active)
#pragma unroll
            for (int w = h; w < h + V; ++w) {
                const int i = w * kGroups + T.g;
                if (w0 + i < nk) {
                    const dc v = cmul(ld2(T.ph, w0 - p0 + i), dc{tr[w], ti[w]});
                    T.re[(i - h * kGroups) * 64 + T.lane] = v.r;
                    T.im[(i - h * kGroups) * 64 + T.lane] = v.i;
                }
            }
        __syncthreads();
        if (T.g < 2) {
            const double* v = (T.g ? T.im : T.re) + T.lane;
            const int cnt = min(V * kGroups, nk - w0 - h * kGroups);
            if (cnt == V * kGroups) {
#pragma unroll
                for (int i = 0; i < V * kGroups; ++i) sum += v[64 * i];
            } else {
                for (int i = 0; i < cnt; ++i) sum += v[64 * i];
            }
        }
    }
}

// U(p) (+)= sum over spheres and waves, 64 pixels a block and the waves of a
// sphere over its wavefronts, kWaves at a time in registers; the c_l of the
// block's pixels sit in LDS, formed once per sphere (per round of waves beyond
// cap orders).  The terms are summed in the reference's order: by wave, then
// by sphere.  With kSplit, blockIdx.y is a sphere, whose sum goes to part.
// Bound by FP64 issue: 11 operations per (pixel, sphere, wave, order) of which
// none may be contracted, the divide's two FMAs apart; 62 to 67 % of the
// issue rate (39e12 a second) on 192 x 192 pixels, 6 spheres of 16 orders or
// so, 200 waves: 0.38 ms, where a kernel that read the c_l from memory for
// every wave took 3.2 (6 launches) and one that formed them for every wave
// more.  8 waves a wavefront and 3 blocks a CU (84 bytes of spills outside
// the loops) against 2: 1537 and 1631 us for four such images.
template <bool kSplit>
__global__ __launch_bounds__(kThreads, 3) void us_series64_kernel(
    QuadArg q, int uR, int vR, d3 f, double kmag, UsSphereBatch batch, int ns,
    const double2* __restrict__ A, const double2* __restrict__ B,
    const double* __restrict__ waves, int nk, double sA, int cap, double* __restrict__ part,
    double* __restrict__ U, int accumulate) {
    extern __shared__ double us64_lds[];
    const int npix = uR * vR;
    Block T;
    T.g = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    T.lane = (int)threadIdx.x & 63;
    T.re = us64_lds;
    T.im = T.re + kGroups * kSum * 64;
    T.ph = (double2*)(T.im + kGroups * kSum * 64);
    T.step = (StepConst*)(T.ph + kPhases);
    T.c = (double2*)(T.step + cap);
    T.cap = cap;
    const int pix = blockIdx.x * 64 + T.lane;
    const int iv = min(pix, npix - 1) / uR, iu = min(pix, npix - 1) - iv * uR;
    const d3 p = quad_at(q, (double)iu / (double)uR, (double)iv / (double)vR);
    double acc = 0.0;   // of the part that the wavefront sums
    if (!kSplit && accumulate && T.g < 2 && pix < npix) acc = U[2 * (size_t)pix + T.g];
    for (int s = kSplit ? (int)blockIdx.y : 0; s < (kSplit ? (int)blockIdx.y + 1 : ns); ++s) {
        const SphereDev& S = batch.s[s];
        const d3 ps = mk(S.p);
        d3 r = sub(p, ps);
        Radial R;
        const double d = len(r);
        R.locate(d, kmag, S);
        r = R.kind == 2 ? d3{0.0, 0.0, 0.0} : norm(r);
        const d3 c = sub(ps, f);
        T.A = A + S.coeff_off;
        T.B = B + S.coeff_off;
        T.Nl = S.Nl;
        double sum = 0.0;
        for (int p0 = 0; p0 < nk; p0 += kPhases) {
            __syncthreads();   // the last phases and c_l are used
            const int p1 = min(p0 + kPhases, nk);
            // (the last threads, whose wavefronts have no chain of hold_orders)
            for (int w = p0 + kThreads - 1 - (int)threadIdx.x; w < p1; w += kThreads) {
                const dc e = cscl(cexp_i(kmag * dot(mk(waves + 3 * w), c)), sA);
                T.ph[w - p0] = make_double2(e.r, e.i);
            }
            if (p0 == 0 && T.Nl < cap) hold_orders(T, R, 0, T.Nl + 1);
            __syncthreads();
            int w = p0;
            for (; w + kGroups * (kWaves / 2) < p1; w += kGroups * kWaves)
                wave_round<kWaves>(T, R, r, waves, w, p0, p1, sum);
            for (; w + kGroups < p1; w += 2 * kGroups)
                wave_round<2>(T, R, r, waves, w, p0, p1, sum);
            for (; w < p1; w += kGroups) wave_round<1>(T, R, r, waves, w, p0, p1, sum);
        }
        if (kSplit) {
            if (T.g < 2 && pix < npix)
                part[2 * ((size_t)batch.slot[s] * npix + pix) + T.g] = sum;
        } else {
            acc = acc + sum;
        }
    }
    if (!kSplit && T.g < 2 && pix < npix) U[2 * (size_t)pix + T.g] = acc;
}

// U (+)= the spheres' sums, in order
__global__ void us_combine64_kernel(int n, int ns, const double* __restrict__ part,
                                    double* __restrict__ U, int accumulate) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double acc = accumulate ? U[i] : 0.0;
    for (int s = 0; s < ns; ++s) acc = acc + part[(size_t)s * n + i];
    U[i] = acc;
}

// The few-wave form: a thread a pixel, W >= nk waves of a sphere in registers,
// the radial chains run beside the waves' own.  The same operations in the same
// order as us_series64_kernel, whose blocks give a pixel's chains and its waves
// a wavefront each and leave most of them idle where there are few waves.
// Bound by FP64 issue.  One wave and one sphere of 18 orders on 256 x 256
// pixels 11 us (28 in the other form), 512 x 512 20 (85); two spheres of 18 on
// 1024 x 1024 121 (545); one of 116 orders on 256 x 256 29 (146); four waves, one
// of 329 orders on 256 x 256 107 (365).
template <int W>
__global__ __launch_bounds__(kThreads) void us_few64_kernel(
    QuadArg q, int uR, int vR, d3 f, double kmag, UsSphereBatch batch, int ns,
    const double2* __restrict__ A, const double2* __restrict__ B,
    const double* __restrict__ waves, int nk, double sA, double2* __restrict__ U, int accumulate) {
    __shared__ double2 ph[W];
    const int npix = uR * vR;
    const int pix = blockIdx.x * kThreads + (int)threadIdx.x;
    const int at = min(pix, npix - 1), iv = at / uR, iu = at - iv * uR;
    const d3 p = quad_at(q, (double)iu / (double)uR, (double)iv / (double)vR);
    dc acc = {0.0, 0.0};
    if (accumulate) acc = ld2(U, at);
    for (int s = 0; s < ns; ++s) {
        const SphereDev& S = batch.s[s];
        const d3 ps = mk(S.p), c = sub(ps, f);
        d3 r = sub(p, ps);
        const double d = len(r), kd = kmag * d;
        const dc knd = cscl(dc{S.n[0], S.n[1]}, kd);
        r = norm(r);
        const bool inside = d <= S.a, centre = inside && knd.r < (double)kEpsFloat;
        const double2* const C = (inside ? A : B) + S.coeff_off;
        __syncthreads();   // the last sphere's phases are used
        if ((int)threadIdx.x < nk) {
            const dc e = cscl(cexp_i(kmag * dot(mk(waves + 3 * threadIdx.x), c)), sA);
            ph[threadIdx.x] = make_double2(e.r, e.i);
        }
        __syncthreads();
        double x[W], P0[W], P1[W], tr[W], ti[W];
#pragma unroll
        for (int w = 0; w < W; ++w) {
            x[w] = dot(mk(waves + 3 * min(w, nk - 1)), r);
            P0[w] = 1.0;
            P1[w] = x[w];
        }
        auto first = [&](dc c0, dc c1) {
#pragma unroll
            for (int w = 0; w < W; ++w) {
                tr[w] = 0.0 + c0.r;
                ti[w] = 0.0 + c0.i;
                tr[w] += c1.r * x[w];
                ti[w] += c1.i * x[w];
            }
        };
        auto order = [&](int l, dc cl) {
            const double a = (double)(2 * l - 1), b = (double)(l - 1), n = (double)l, inv = 1.0 / n;
#pragma unroll
            for (int w = 0; w < W; ++w) {
                const double Pn = div_int(a * x[w] * P1[w] - b * P0[w], n, inv);
                P0[w] = P1[w];
                P1[w] = Pn;
                tr[w] += cl.r * Pn;
                ti[w] += cl.i * Pn;
            }
        };
        if (centre) {   // calc_Ui: A_0 for every wave
            const dc c0 = ld2(C, 0);
#pragma unroll
            for (int w = 0; w < W; ++w) {
                tr[w] = c0.r;
                ti[w] = c0.i;
            }
        } else if (inside) {
            dc j[2];
            ref::init_jc(knd, j);
            first(cmul(ld2(C, 0), j[0]), cmul(ld2(C, 1), j[1]));
            for (int l = 2; l <= S.Nl; ++l) {
                ref::shift_jc(l, knd, j);
                order(l, cmul(ld2(C, l), j[1]));
            }
        } else {
            double j[2], y[2];
            ref::init_j(kd, j);
            ref::init_y(kd, y);
            first(cmul(ld2(C, 0), dc{j[0], y[0]}), cmul(ld2(C, 1), dc{j[1], y[1]}));
            for (int l = 2; l <= S.Nl; ++l) {
                ref::shift_j(l, kd, j);
                ref::shift_y(l, kd, y);
                order(l, cmul(ld2(C, l), dc{j[1], y[1]}));
            }
        }
        dc sum = {0.0, 0.0};
#pragma unroll
        for (int w = 0; w < W; ++w)
            if (w < nk) sum = cadd(sum, cmul(ld2(ph, w), dc{tr[w], ti[w]}));
        acc = cadd(acc, sum);
    }
    if (pix < npix) U[pix] = make_double2(acc.r, acc.i);
}

__global__ void clear_c64(double2* U, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) U[i] = make_double2(0.0, 0.0);
}
__global__ void clear_c32(float2* U, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) U[i] = make_float2(0.f, 0.f);
}
// U (+)= the complex128 field W rounded to complex64
__global__ void narrow_add_kernel(const double2* __restrict__ W, float2* __restrict__ U, int n,
                                  int accumulate) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double2 w = W[i];
    float2 v = make_float2(0.f, 0.f);
    if (accumulate) v = U[i];
    U[i] = make_float2(v.x + (float)w.x, v.y + (float)w.y);
}

SphereDev to_dev(const bimsim_sphere& S) {
    SphereDev d;
    for (int c = 0; c < 3; ++c) d.p[c] = S.p[c];
    d.a = S.a;
    d.n[0] = S.n[0];
    d.n[1] = S.n[1];
    d.Nl = S.Nl;
    d.coeff_off = S.coeff_off;
    return d;
}

// Both FP64 precisions.  A sphere of its own per block, the sums added up by a
// launch of their own, where one block per 64 pixels would leave CUs idle or
// end in a long last wave (up to kSplitBlocks of them), largest spheres first;
// a call that cannot have the sums' scratch loops over the spheres instead,
// with the same operations.
constexpr int kSplitBlocks = 4096;

// Whether a call takes the few-wave form: up to two waves where the pixels are
// more than two wavefronts a CU (one wave, 192 x 192: one sphere 12 us and 19
// in the other form, four of 39 orders 64 and 68; 144 x 144: 13 and 15, 64 and
// 48), three or four where they are four (256 x 256: 17 and 28, 47 and 60; 224
// x 224, four spheres: 107 and 95).
bool few_waves64(const bimsim_ctx* ctx, int npix, int nk) {
    return (nk <= 2 && npix > 128 * ctx->cu_count) || (nk <= 4 && npix >= 256 * ctx->cu_count);
}

int us_series64(bimsim_ctx* ctx, const QuadArg& q, int uR, int vR, d3 f, double kmag,
                const bimsim_sphere* spheres, int ns, const double2* A, const double2* B,
                const double* waves, int nk, double sA, int lmax, double* U, int accumulate) {
    const int npix = uR * vR, blocks = (npix + 63) / 64;
    const int cap = std::min(lmax + 1, kOrders);
    const size_t lds = (size_t)kSumBytes + sizeof(double2) * kPhases +
                       (size_t)cap * (sizeof(StepConst) + 64 * sizeof(double2));
    const bool few = few_waves64(ctx, npix, nk);
    void* part = nullptr;
    if (!few && ns > 1 && blocks <= kSplitBlocks)
        part = scratch_try(ctx, kSlotSums, sizeof(double2) * (size_t)std::min(ns, kUsBatch) * npix);
    for (int s0 = 0; s0 < ns; s0 += kUsBatch) {
        const int cnt = std::min(kUsBatch, ns - s0), add = (s0 > 0 || accumulate) ? 1 : 0;
        UsSphereBatch b{};
        for (int i = 0; i < cnt; ++i) b.slot[i] = i;
        if (part)
            std::stable_sort(b.slot, b.slot + cnt, [&](int x, int y) {
                return spheres[s0 + x].Nl > spheres[s0 + y].Nl;
            });
        for (int i = 0; i < cnt; ++i) b.s[i] = to_dev(spheres[s0 + b.slot[i]]);
        if (few) {
            auto launch = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3((npix + kThreads - 1) / kThreads), dim3(kThreads),
                                   0, ctx->stream, q, uR, vR, f, kmag, b, cnt, A, B, waves, nk, sA,
                                   (double2*)U, add);
            };
            if (nk == 1) launch(us_few64_kernel<1>);
            else if (nk == 2) launch(us_few64_kernel<2>);
            else launch(us_few64_kernel<4>);
        } else if (part) {
            hipLaunchKernelGGL(us_series64_kernel<true>, dim3(blocks, cnt), dim3(kThreads), lds,
                               ctx->stream, q, uR, vR, f, kmag, b, cnt, A, B, waves, nk, sA, cap,
                               (double*)part, U, add);
            hipLaunchKernelGGL(us_combine64_kernel, dim3((2 * npix + kThreads - 1) / kThreads),
                               dim3(kThreads), 0, ctx->stream, 2 * npix, cnt, (const double*)part,
                               U, add);
        } else {
            hipLaunchKernelGGL(us_series64_kernel<false>, dim3(blocks), dim3(kThreads), lds,
                               ctx->stream, q, uR, vR, f, kmag, b, cnt, A, B, waves, nk, sA, cap,
                               (double*)nullptr, U, add);
        }
        BIMSIM_HIP_CHECK(ctx, hipGetLastError());
    }
    return BIMSIM_OK;
}

}  // namespace
}  // namespace bimsim

namespace bimsim {

int us_wide_fp32(bimsim_ctx* ctx, const bimsim_quad* pos, int uR, int vR, const double focus[3],
                 double kmag, const bimsim_sphere* spheres, int ns, const void* A, const void* B,
                 const double* waves, int nk, double subA, float2* U, int accumulate) {
    const int npix = uR * vR;
    void* wide = nullptr;
    BIMSIM_TRY(scratch_get(ctx, kSlotWide, sizeof(double2) * (size_t)npix, &wide));
    BIMSIM_TRY(bimsim_nf_us(ctx, pos, uR, vR, focus, kmag, spheres, ns, A, B, waves, nk, subA,
                            BIMSIM_FP64, BIMSIM_QUIRKS_REF, wide, 0));
    hipLaunchKernelGGL(narrow_add_kernel, dim3((npix + kThreads - 1) / kThreads), dim3(kThreads), 0,
                       ctx->stream, (const double2*)wide, U, npix, accumulate ? 1 : 0);
    BIMSIM_HIP_CHECK(ctx, hipGetLastError());
    return BIMSIM_OK;
}

}  // namespace bimsim

using namespace bimsim;

extern "C" int bimsim_nf_us(bimsim_ctx* ctx, const bimsim_quad* pos, int uR, int vR,
                            const double focus[3], double kmag, const bimsim_sphere* spheres,
                            int ns, const void* A, const void* B, const double* waves, int nk,
                            double subA, int prec, int quirks, void* U, int accumulate) {
    if (!ctx) return BIMSIM_E_INVALID;
    BIMSIM_CHECK_ARG(ctx, pos && focus && U, "null pointer argument");
    BIMSIM_CHECK_ARG(ctx, uR > 0 && vR > 0 && (long long)uR * vR <= (1LL << 28),
                     "slice resolution must be positive and at most 2^28 pixels");
    BIMSIM_CHECK_ARG(ctx, ns >= 0 && nk > 0, "ns must be >= 0 and nk > 0");
    BIMSIM_CHECK_ARG(ctx, prec >= BIMSIM_FP64_PARITY && prec <= BIMSIM_FP32_FAST, "unknown precision");
    BIMSIM_CHECK_ARG(ctx, kmag > 0.0 && std::isfinite(kmag), "kmag must be positive");
    if (!quirks)
        return set_error(ctx, BIMSIM_E_UNSUPPORTED,
                         "scattered-field series without the reference recurrences is not built");
    BIMSIM_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    const int npix = uR * vR;
    const int pix_blocks = (npix + kThreads - 1) / kThreads;
    if (ns == 0) {
        if (!accumulate) {
            if (prec == BIMSIM_FP32_FAST)
                hipLaunchKernelGGL(clear_c32, dim3(pix_blocks), dim3(kThreads), 0, ctx->stream, (float2*)U, npix);
            else
                hipLaunchKernelGGL(clear_c64, dim3(pix_blocks), dim3(kThreads), 0, ctx->stream, (double2*)U, npix);
            BIMSIM_HIP_CHECK(ctx, hipGetLastError());
        }
        return BIMSIM_OK;
    }
    BIMSIM_CHECK_ARG(ctx, spheres && A && B && waves, "null sphere/coefficient/wave pointer");
    int lmax = 0;
    for (int s = 0; s < ns; ++s) {
        BIMSIM_CHECK_ARG(ctx, spheres[s].Nl >= 1 && spheres[s].a > 0.0 && spheres[s].coeff_off >= 0,
                         "sphere needs Nl >= 1, a > 0, coeff_off >= 0");
        lmax = std::max(lmax, spheres[s].Nl);
    }
    const QuadArg q = to_quad(*pos);
    const d3 f = mk(focus);
    // ptype scale = (1.0f/nk) (nfScalarUs.cu:461): float arithmetic
    const double sA = (double)(1.0f / (float)nk) * subA;
    const int tmr = timer_begin(ctx, kStageUs);
    if (prec != BIMSIM_FP32_FAST) {
        BIMSIM_TRY(us_series64(ctx, q, uR, vR, f, kmag, spheres, ns, (const double2*)A,
                               (const double2*)B, waves, nk, sA, lmax, (double*)U, accumulate));
    } else if (series_capacity(lmax + 1) < 0) {
        // orders beyond the FP32 series kernels: the FP64 form, rounded
        timer_end(ctx, tmr);
        return us_wide_fp32(ctx, pos, uR, vR, focus, kmag, spheres, ns, A, B, waves, nk, subA,
                            (float2*)U, accumulate);
    } else {
        // FP32 series: a batch of one instance
        SeriesBatch batch;
        SeriesInst I{};
        I.q = q;
        I.f = f;
        I.kmag = kmag;
        I.sA = sA;
        I.uR = uR;
        I.vR = vR;
        I.s_begin = 0;
        I.ns = ns;
        I.nk = nk;
        I.accumulate = accumulate ? 1 : 0;
        batch.inst.push_back(I);
        for (int s = 0; s < ns; ++s) {
            SeriesSph S{};
            S.s = to_dev(spheres[s]);
            S.inst = 0;
            batch.sph.push_back(S);
        }
        const SeriesPlan* plan = nullptr;
        BIMSIM_TRY(series_cached_plan(ctx, batch, waves, (const double2*)A, (const double2*)B, &plan));
        BIMSIM_TRY(series_plan_launch(ctx, *plan, waves, (const double2*)A, (const double2*)B,
                                     (float2*)U));
    }
    timer_end(ctx, tmr);
    return BIMSIM_OK;
}
