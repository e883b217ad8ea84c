"""The Monte-Carlo incident field from the nodes of its tiles and from its
pixels: edges of tiles, the node counts' limits, waves that are no unit
vectors, and the wide tiles of many images."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def waves_of(nk, scale, seed=3):
    rng = np.random.default_rng(seed)
    k = rng.normal(size=(nk, 3))
    return scale * k / np.linalg.norm(k, axis=1)[:, None]


# width / N against the wavelength pi: 31.5 kh = 63 width / N sets the nodes
# per edge (16, 24, 32 and 40 at kh = 3.2, 7.5, 13, 20); waves about twice as
# many as the nodes, and about a chunk of 32
@pytest.mark.parametrize("uR,vR,pitch,nk,scale", [
    (1, 1, 0.1, 1, 1.0), (64, 64, 0.01, 300, 1.0), (65, 63, 0.05, 31, 1.0),
    (63, 130, 0.05, 33, 1.0), (128, 64, 0.051, 64, 1.0), (70, 70, 0.118, 97, 1.0),
    (70, 70, 0.12, 97, 1.0), (96, 65, 0.206, 200, 1.0), (96, 65, 0.21, 200, 1.0),
    (100, 100, 0.3, 80, 1.0), (100, 100, 0.33, 90, 1.0), (100, 100, 1.2, 90, 1.0),
    (66, 66, 0.01, 9, 1.0), (66, 66, 0.05, 64, 7.0), (66, 66, 0.05, 64, 0.25)])
def test_matches_oracle(pkg, ctx, orc, uR, vR, pitch, nk, scale):
    kmag, subA = 2.0, 0.8
    q = pkg.Quad.xy(1.0)
    q.A[:] = [-3.0, 1.0, 0.4]
    q.X[:] = [pitch * uR, 0.02, 0.0]
    q.Y[:] = [0.0, 0.9 * pitch * vR, 0.1]
    k = waves_of(nk, scale)
    focus = (0.3, -0.1, 0.2)
    want = orc.nf_uf_mc(q, uR, vR, focus, kmag, k, subA).ravel()
    U = torch.full((uR * vR + 5,), 9.0, dtype=torch.complex64, device="cuda")
    ctx.nf_uf_mc(q, uR, vR, focus, kmag, torch.as_tensor(k).cuda(), subA, U, prec=pkg.FP32_FAST)
    got = U.cpu().numpy()
    assert (got[uR * vR:] == 9.0).all()
    # every wave within 3e-8 of its weight by interpolation, 2e-7 by its
    # factors and their product, and half an ulp a partial sum
    weight = subA / nk
    bound = weight * (3e-7 * nk + 6e-8 * nk * np.sqrt(nk))
    assert np.abs(got[:uR * vR] - want).max() <= bound


def test_waves_that_are_not_numbers_stay_so(pkg, ctx):
    k = waves_of(64, 1.0)
    k[17, 0] = np.nan
    U = torch.zeros(70 * 70, dtype=torch.complex64, device="cuda")
    ctx.nf_uf_mc(pkg.Quad.xy(2.0), 70, 70, (0.0, 0.0, 0.0), 2.0, torch.as_tensor(k).cuda(), 1.0, U,
                 prec=pkg.FP32_FAST)
    assert bool(torch.isnan(U.real).all())


@pytest.mark.parametrize("N,width", [(2900, 30.0), (2944, 400.0), (2900, 900.0)])
def test_wide_tiles(pkg, ctx, N, width):
    """A slice of 512 or more tiles of 128 pixels: nodes of those, of their
    quarters, and pixels, against slices of its rows."""
    nk = 120
    w = torch.as_tensor(waves_of(nk, 1.0)).cuda()
    U = torch.empty(N * N, dtype=torch.complex64, device="cuda")
    q = pkg.Quad.xy(width)
    ctx.nf_uf_mc(q, N, N, (0.0, 0.0, 0.0), 2.0, w, 1.0, U, prec=pkg.FP32_FAST)
    U = U.view(N, N)
    for rows in (0, 127, N - 70):
        part = pkg.Quad.xy(width)
        part.A[1] = part.A[1] + width * rows / N
        part.Y[1] = width * 70 / N
        P = torch.empty(70 * N, dtype=torch.complex64, device="cuda")
        ctx.nf_uf_mc(part, N, 70, (0.0, 0.0, 0.0), 2.0, w, 1.0, P, prec=pkg.FP32_FAST)
        # twice the bound above
        assert float((U[rows:rows + 70] - P.view(70, N)).abs().max()) <= 2 * (3e-7 + 6e-8 * nk ** 0.5)
