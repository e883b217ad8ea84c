"""The detector at FFT lengths with and without a compiled stage plan, with
supersampling, padding and zero filling, against numpy's FFT; and batches
whose instances share an image."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def expected(U, Uf, N, fill, du, NAin, NAout, lam, padding, Nd, ss):
    """(D, Di) in FP64: numpy FFT, the band-pass with the reference's
    negative-frequency index -(M-1-i), the crop and the mean of |.|^2."""
    M = N * fill
    i = np.arange(M)
    f = np.where(i <= M // 2, i, -(M - 1 - i)) * (du / fill)
    r = np.sqrt(f[None, :] ** 2 + f[:, None] ** 2)
    keep = ~((r < NAin / lam) | (r > NAout / lam))
    out = []
    for F in (U, Uf):
        G = np.zeros((M, M), dtype=np.complex128)
        G[:N, :N] = F.reshape(N, N)
        G = np.fft.ifft2(np.fft.fft2(G) * keep)
        o = padding * Nd * ss
        G = np.abs(G[o: o + Nd * ss, o: o + Nd * ss]) ** 2
        out.append(G.reshape(Nd, ss, Nd, ss).mean(axis=(1, 3)).ravel())
    return out


def fields(N, seed):
    rng = np.random.default_rng(seed)
    return [rng.normal(size=N * N) + 1j * rng.normal(size=N * N) for _ in range(2)]


# lengths: one and two elements, one stage of each radix, odd powers, the
# radices mixed, a compiled length beside them, rows of more than 1024
@pytest.mark.parametrize("N", [1, 2, 3, 5, 8, 25, 27, 45, 60, 64, 125, 250, 320, 375, 640, 720,
                               1000, 1280])
@pytest.mark.parametrize("prec", [1, 2])
def test_detector_at_any_length(pkg, ctx, N, prec):
    cd, rd = (torch.complex64, torch.float32) if prec == 2 else (torch.complex128, torch.float64)
    U, Uf = fields(N, N)
    lam, L = 4.0, 100.0
    cases = [(0, N, 1, 1)]
    if N % 2 == 0:
        cases.append((0, N // 2, 2, 1))
    if N % 3 == 0:
        cases.append((1, N // 3, 1, 1))
    if N <= 375:
        cases += [(0, N, 1, 2), (0, N, 1, 3)]
    # FP32: about log2(M^2) roundings of 6e-8 each way on a random field
    tol = 2e-6 if prec == 2 else 1e-13
    for padding, Nd, ss, fill in cases:
        ud, ufd = (torch.as_tensor(F).to(cd).cuda() for F in (U, Uf))
        D, Di, Ab = (torch.zeros(Nd * Nd, dtype=rd, device="cuda") for _ in range(3))
        # a pass band of part of the spectrum (everything where there is little)
        na = (0.0, 1.0 * lam / L * max(1, N // 3))
        if fill > 1:
            ctx.detector_zero_filled(ud, ufd, N, N, fill, 1 / L, 1 / L, *na, lam, D, Di, Ab,
                                     prec=prec)
        else:
            ctx.detector(ud, ufd, N, N, 1 / L, 1 / L, *na, lam, padding, Nd, ss, D, Di, Ab,
                         prec=prec, write_filtered=False)
        want = expected(U, Uf, N, fill, 1 / L, *na, lam, padding, Nd, ss)
        for got, w in ((D, want[0]), (Di, want[1])):
            got = got.cpu().numpy().astype(np.float64)
            assert np.linalg.norm(got - w) <= tol * np.linalg.norm(w), (N, padding, ss, fill)
        if fill == 1:   # the filtered fields left in place give the same images
            D2, Di2 = torch.zeros_like(D), torch.zeros_like(Di)
            ctx.detector(ud, ufd, N, N, 1 / L, 1 / L, *na, lam, padding, Nd, ss, D2, Di2, None,
                         prec=prec, write_filtered=True)
            assert (D2 - D).norm() <= tol * D.norm() and (Di2 - Di).norm() <= tol * Di.norm()
            o = padding * Nd * ss
            F = ud.reshape(N, N)[o: o + Nd * ss, o: o + Nd * ss].abs().to(torch.float64) ** 2
            F = F.reshape(Nd, ss, Nd, ss).mean(dim=(1, 3)).reshape(-1)
            assert (F - D.to(torch.float64)).norm() <= 2 * tol * F.norm()


@pytest.mark.parametrize("uR,vR", [(60, 90), (128, 45), (64, 512), (375, 96)])
@pytest.mark.parametrize("prec", [1, 2])
def test_rectangular_fields(pkg, ctx, uR, vR, prec):
    """Rows and columns of different lengths, with a compiled plan or without."""
    cd, rd = (torch.complex64, torch.float32) if prec == 2 else (torch.complex128, torch.float64)
    rng = np.random.default_rng(uR)
    U, Uf = [rng.normal(size=(vR, uR)) + 1j * rng.normal(size=(vR, uR)) for _ in range(2)]
    lam, Lu, Lv, ss = 4.0, 100.0, 130.0, 1 if uR % 2 else 2
    Nd = min(uR, vR) // ss
    na = (0.02, 0.3 * lam * min(uR / Lu, vR / Lv))

    def axis(n, L):
        i = np.arange(n)
        return np.where(i <= n // 2, i, -(n - 1 - i)) / L

    f = np.sqrt(axis(uR, Lu)[None, :] ** 2 + axis(vR, Lv)[:, None] ** 2)
    keep = ~((f < na[0] / lam) | (f > na[1] / lam))
    ud, ufd = (torch.as_tensor(F.ravel()).to(cd).cuda() for F in (U, Uf))
    D, Di = (torch.zeros(Nd * Nd, dtype=rd, device="cuda") for _ in range(2))
    ctx.detector(ud, ufd, uR, vR, 1 / Lu, 1 / Lv, *na, lam, 0, Nd, ss, D, Di, None, prec=prec,
                 write_filtered=False)
    tol = 2e-6 if prec == 2 else 1e-13
    for got, F in ((D, U), (Di, Uf)):
        G = np.abs(np.fft.ifft2(np.fft.fft2(F) * keep)[: Nd * ss, : Nd * ss]) ** 2
        want = G.reshape(Nd, ss, Nd, ss).mean(axis=(1, 3)).ravel()
        got = got.cpu().numpy().astype(np.float64)
        assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want)


@pytest.mark.parametrize("prec", [1, 2])
def test_one_transform_size_of_different_fields(pkg, ctx, prec):
    """Zero-filled and plain instances whose FFTs are of one size share their
    launches: fields of 50, 100 and 25 samples at 100 points, and two others."""
    import bimsim_amd.pipeline as P
    import bimsim_amd.workloads as W
    insts = []
    for N, fill in ((50, 2), (100, 0), (25, 4), (40, 0), (50, 0)):
        i = W.config(1, N=N, nk=20)
        i["zero_fill"] = fill
        insts.append(i)
    waves = [W.mc_waves(i, pkg.mc_sample_na) for i in insts]
    arr, spheres, Wv, n = P.batch_tables(insts, waves)
    rd = torch.float32 if prec == 2 else torch.float64
    D, Di, Ab = (torch.zeros(n, dtype=rd, device="cuda") for _ in range(3))
    b = ctx.batch(arr, spheres, torch.as_tensor(Wv.ravel()).cuda(), D, Di, Ab, prec=prec)
    b.launch()
    at, tol = 0, 2e-6 if prec == 2 else 1e-13
    for inst, w in zip(insts, waves):
        one = P.simulate(ctx, inst, torch.as_tensor(w).cuda(), prec)
        m = inst["Nd"] ** 2
        for got, want in ((D, one.D), (Di, one.Di)):
            assert (got[at: at + m] - want).norm() <= tol * want.norm(), inst["N"]
        at += m
    b.close()


def test_length_with_another_factor_is_refused(pkg, ctx):
    N = 28
    U = torch.zeros(N * N, dtype=torch.complex128, device="cuda")
    D, Di = (torch.zeros(N * N, dtype=torch.float64, device="cuda") for _ in range(2))
    with pytest.raises(pkg.BimsimError) as e:
        ctx.detector(U, U, N, N, 0.01, 0.01, 0.0, 0.5, 4.0, 0, N, 1, D, Di, prec=1)
    assert e.value.code == pkg.E_UNSUPPORTED


@pytest.mark.parametrize("N", [48, 64, 100])
@pytest.mark.parametrize("prec", [1, 2])
def test_instances_sharing_an_image_add_up(pkg, ctx, N, prec):
    """Three sources on one image and a fourth instance on its own, at lengths
    with and without a compiled plan: the shared image holds the sum."""
    import bimsim_amd.pipeline as P
    import bimsim_amd.workloads as W
    base = W.config(2, N=N, nk=20)
    insts = []
    for f in ((0.0, 0.0, 0.0), (3.0, -2.0, 0.0), (-4.0, 5.0, 0.0), (1.0, 1.0, 0.0)):
        i = dict(base)
        i["focus"] = f
        insts.append(i)
    waves = [W.mc_waves(i, pkg.mc_sample_na) for i in insts]
    singles = [P.simulate(ctx, i, torch.as_tensor(w).cuda(), prec) for i, w in zip(insts, waves)]
    arr, spheres, Wv, _ = P.batch_tables(insts, waves)
    for k, off in enumerate((0, 0, 0, N * N)):
        arr[k].image_off = off
    rd = torch.float32 if prec == 2 else torch.float64
    D = torch.full((2 * N * N,), 7.0, dtype=rd, device="cuda")
    Di, Ab = torch.full_like(D, 7.0), torch.empty_like(D)
    b = ctx.batch(arr, spheres, torch.as_tensor(Wv.ravel()).cuda(), D, Di, Ab, prec=prec)
    for _ in range(2):
        b.launch()
    tol = 2e-6 if prec == 2 else 1e-13
    for got, name in ((D, "D"), (Di, "Di")):
        one = [getattr(s, name).double() for s in singles]
        want = torch.cat([one[0] + one[1] + one[2], one[3]])
        assert (got.double() - want).norm() <= tol * want.norm()
    b.close()
