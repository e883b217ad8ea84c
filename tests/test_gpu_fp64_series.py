"""The FP64 scattered field where its rounds of waves, its orders in LDS and its
split over spheres have edges: against the oracle, and one way against another
bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def setup(pkg, ns, nk, ka, kmag=1.5, seed=5):
    """ns spheres, the first of size ka and the others smaller, and nk waves."""
    rng = np.random.default_rng(seed)
    spheres, off = [], 0
    for i in range(ns):
        a = ka / kmag / (1.0 + 0.4 * i)
        p = (0.0, 0.0, 0.0) if i == 0 else tuple(rng.uniform(-1.0, 1.0, 3) * 3.0 * ka / kmag)
        spheres.append(dict(p=p, a=a, n=complex(1.3 + 0.02 * i, 0.01 * i), coeff_off=off,
                            Nl=pkg.sphere_order(a, 2 * np.pi / kmag)))
        off += spheres[-1]["Nl"] + 1
    k = rng.normal(size=(nk, 3))
    return spheres, off, kmag, k / np.linalg.norm(k, axis=1)[:, None]


def field(pkg, ctx, spheres, A, B, kmag, waves, uR, vR, width, prec, U=None):
    out = torch.empty(uR * vR, dtype=torch.complex128, device="cuda") if U is None else U.clone()
    ctx.nf_us(pkg.Quad.xy(width), uR, vR, (0.1, -0.2, 0.3), kmag, spheres, A, B, waves, 0.7, out,
              prec=prec, accumulate=U is not None)
    return out


def coefficients(ctx, spheres, off, kmag):
    A = torch.empty(off, dtype=torch.complex128, device="cuda")
    B = torch.empty_like(A)
    ctx.mie_coeffs(spheres, kmag, A, B)
    return A, B


# waves about 1, 4, 8, 16, 32 and 128 a round; orders about the 112 held in
# LDS; pixels that are no multiple of 64
@pytest.mark.parametrize("ns,nk,ka,uR,vR", [
    (1, 1, 0.3, 1, 1), (1, 3, 2.0, 64, 1), (2, 4, 2.0, 13, 5), (2, 5, 3.0, 65, 1),
    (1, 16, 4.0, 9, 7), (3, 17, 2.0, 8, 8), (1, 33, 9.0, 16, 9), (2, 127, 3.0, 7, 7),
    (1, 128, 3.0, 10, 10), (1, 129, 3.0, 10, 10), (33, 9, 2.0, 9, 9), (1, 20, 91.0, 11, 6),
    (1, 7, 93.0, 11, 6), (2, 41, 190.0, 8, 8)])
def test_matches_oracle(pkg, ctx, orc, ns, nk, ka, uR, vR):
    spheres, off, kmag, k = setup(pkg, ns, nk, ka)
    A, B = coefficients(ctx, spheres, off, kmag)
    waves = torch.as_tensor(k).cuda()
    width = 5.0 * ka / kmag
    want = orc.nf_us(pkg.Quad.xy(width), uR, vR, (0.1, -0.2, 0.3), kmag, spheres, A.cpu().numpy(),
                     B.cpu().numpy(), k, 0.7).ravel()
    for prec in (pkg.FP64_PARITY, pkg.FP64):
        got = field(pkg, ctx, spheres, A, B, kmag, waves, uR, vR, width, prec).cpu().numpy()
        assert np.abs(got - want).max() <= 1e-10 * np.abs(want).max()


def test_split_over_spheres_keeps_the_bits(pkg, ctx):
    """Spheres in one call (a block each, sums added up after), one call a
    sphere, and a captured call of a context that has no scratch yet."""
    spheres, off, kmag, k = setup(pkg, 35, 21, 6.0)
    A, B = coefficients(ctx, spheres, off, kmag)
    waves = torch.as_tensor(k).cuda()
    U0 = torch.randn(2, 33 * 21, dtype=torch.float64, device="cuda").T.contiguous()
    U0 = torch.view_as_complex(U0)
    together = field(pkg, ctx, spheres, A, B, kmag, waves, 33, 21, 30.0, pkg.FP64, U0)
    apart = U0
    for s in spheres:
        apart = field(pkg, ctx, [s], A, B, kmag, waves, 33, 21, 30.0, pkg.FP64, apart)
    assert torch.equal(together, apart)

    side = torch.cuda.Stream()
    c = pkg.Context(0, stream=side.cuda_stream)
    out = U0.clone()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        c.nf_us(pkg.Quad.xy(30.0), 33, 21, (0.1, -0.2, 0.3), kmag, spheres, A, B, waves, 0.7, out,
                prec=pkg.FP64, accumulate=True)
    for _ in range(3):
        out.copy_(U0)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, together)
    del g
    c.close()


def test_slices_beyond_the_split(pkg, ctx):
    """More blocks of pixels than a split takes: the same bits as its rows in
    calls that are split."""
    spheres, off, kmag, k = setup(pkg, 2, 5, 2.0)
    A, B = coefficients(ctx, spheres, off, kmag)
    waves = torch.as_tensor(k).cuda()
    n, rows = 64, 4097
    q = pkg.Quad.xy(20.0)
    whole = torch.empty(rows * n, dtype=torch.complex128, device="cuda")
    ctx.nf_us(q, n, rows, (0.0, 0.0, 0.0), kmag, spheres, A, B, waves, 0.7, whole, prec=pkg.FP64)
    # a slice whose first row is the whole one's row 0
    first = torch.empty(n, dtype=torch.complex128, device="cuda")
    ctx.nf_us(q, n, 1, (0.0, 0.0, 0.0), kmag, spheres, A, B, waves, 0.7, first, prec=pkg.FP64)
    assert torch.equal(whole[:n], first)
    # v = j / 4097 of the rows that share v with a slice of 241 (17 241 = 4097)
    part = torch.empty(241 * n, dtype=torch.complex128, device="cuda")
    ctx.nf_us(q, n, 241, (0.0, 0.0, 0.0), kmag, spheres, A, B, waves, 0.7, part, prec=pkg.FP64)
    a, b = whole.view(rows, n)[::17], part.view(241, n)
    assert float((a - b).abs().max()) <= 1e-10 * float(b.abs().max())


# both sides of the few-wave form's limits (more than 128 pixels a CU, or from
# 256 on), spheres that cover part of the slice and one centred on a pixel,
# orders past those the other form holds at a time, more than 32 spheres
@pytest.mark.parametrize("ns,nk,ka,uR,vR", [
    (1, 1, 3.0, 181, 181), (1, 1, 3.0, 182, 182), (3, 2, 2.0, 257, 129), (2, 3, 3.0, 256, 256),
    (1, 4, 93.0, 300, 219), (1, 1, 93.0, 222, 150), (35, 2, 2.0, 200, 165), (1, 5, 3.0, 256, 256)])
def test_few_waves(pkg, ctx, orc, ns, nk, ka, uR, vR):
    spheres, off, kmag, k = setup(pkg, ns, nk, ka)
    A, B = coefficients(ctx, spheres, off, kmag)
    waves = torch.as_tensor(k).cuda()
    width = 5.0 * ka / kmag
    U0 = torch.view_as_complex(torch.randn(uR * vR, 2, dtype=torch.float64, device="cuda"))
    for U in (None, U0):
        got = field(pkg, ctx, spheres, A, B, kmag, waves, uR, vR, width, pkg.FP64, U)
        parity = field(pkg, ctx, spheres, A, B, kmag, waves, uR, vR, width, pkg.FP64_PARITY, U)
        assert torch.equal(got, parity)
        # the first row alone (the same points) takes the other form: the same bits
        row = field(pkg, ctx, spheres, A, B, kmag, waves, uR, 1, width, pkg.FP64,
                    None if U is None else U[:uR])
        assert torch.equal(got[:uR], row)
    want = orc.nf_us(pkg.Quad.xy(width), uR, vR, (0.1, -0.2, 0.3), kmag, spheres, A.cpu().numpy(),
                     B.cpu().numpy(), k, 0.7).ravel()
    got = field(pkg, ctx, spheres, A, B, kmag, waves, uR, vR, width, pkg.FP64).cpu().numpy()
    assert np.abs(got - want).max() <= 1e-10 * np.abs(want).max()
