"""The harmonic scattered field evaluated at nodes of tiles and expanded to
the pixels, against the FP64 form at every pixel: slices of every kind a call
accepts, ragged sizes, spheres on, off and outside the slice.  (That the calls
here take nodes is checked on the host, in test_node_rule.py.)"""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def quad(pkg, A, X, Y):
    q = pkg.Quad()
    q.A[:], q.X[:], q.Y[:] = A, X, Y
    return q


def spheres_of(pkg, lam, rows):
    out, off = [], 0
    for p, a, n in rows:
        s = dict(p=p, a=a, n=n, Nl=pkg.sphere_order(a, lam), coeff_off=off)
        off += s["Nl"] + 1
        out.append(s)
    return out, off


# far spheres (their own nodes are the coarsest tiles'), and 50
# of next to no field that make every call worth its nodes
FAR = ([((200.0 + 20.0 * i, 300.0, 0.0), 3.0, 1.4 + 0.01j) for i in range(9)] +
       [((200.0 + 20.0 * (i % 10), 320.0 + 20.0 * (i // 10), 0.0), 3.0, 1.0 + 1e-5j)
        for i in range(50)])


def both(pkg, ctx, q, uR, vR, lam, rows, nk=20, accumulate=False, seed=0):
    kmag = 2.0 * math.pi / lam
    spheres, n = spheres_of(pkg, lam, rows + FAR)
    A = torch.zeros(n, dtype=torch.complex128, device="cuda")
    B = torch.zeros_like(A)
    ctx.mie_coeffs(spheres, kmag, A, B)
    waves = torch.tensor(pkg.mc_sample_na(nk, (0.0, 0.0, 1.0), 0.1, 0.6, pkg.RNG_SPLITMIX64, seed),
                         dtype=torch.float64).cuda()
    out = []
    for prec, cd in ((pkg.FP64, torch.complex128), (pkg.FP32_FAST, torch.complex64)):
        U = torch.full((uR * vR,), 0.25 - 0.5j, dtype=cd, device="cuda")
        for _ in range(2 if not accumulate else 1):   # the second call reuses the plan
            ctx.nf_us(q, uR, vR, (0.5, -0.25, 0.0), kmag, spheres, A, B, waves, 1.3, U, prec=prec,
                      accumulate=accumulate)
        out.append(U.to(torch.complex128))
    return out + [sum(s["Nl"] + 1 for s in spheres)]


def check(result):
    want, got, terms = result
    err = (got - want).abs()
    rms = float(want.abs().pow(2).mean().sqrt())
    # an FP32 sum of `terms` orders, each addition off by half an ulp at most
    # and either way: 2^-24 sqrt(terms) of the field's rms (1e-6 for 13 spheres
    # of 20 orders), nine times that anywhere, more only where the field itself
    # is larger (near the spheres); an interpolant too coarse, or a tile taken
    # from the wrong place, is off by far more
    tol = 2.0 ** -24 * terms ** 0.5
    assert float(err.norm() / want.norm()) <= tol
    assert float((err / torch.clamp(want.abs(), min=rms)).max()) <= 9 * tol


ROWS = [((0.0, 0.0, 0.0), 5.0, 1.45 + 0.02j), ((-14.0, 9.0, 0.0), 3.0, 1.6 + 0.1j),
        ((17.0, 15.0, 0.0), 2.0, 1.33 + 0.0j), ((40.0, -3.0, 0.0), 4.0, 1.5 + 0.01j)]


# 64 and its neighbours, a last tile of one and of 63 pixels, a prime
@pytest.mark.parametrize("uR,vR", [(256, 256), (320, 192), (257, 320), (383, 449), (512, 130)])
@pytest.mark.parametrize("lam", [2.5, 9.0])
def test_nodes_on_planar_slices(pkg, ctx, uR, vR, lam):
    q = quad(pkg, (-30.0, -25.0, 0.0), (60.0, 0.0, 0.0), (0.0, 50.0, 0.0))
    check(both(pkg, ctx, q, uR, vR, lam, ROWS))


@pytest.mark.parametrize("name,X,Y", [
    ("rotated in the plane", (40.0, 30.0, 0.0), (-30.0, 40.0, 0.0)),
    ("tilted", (50.0, 0.0, 20.0), (0.0, 50.0, -10.0)),
    ("upright", (50.0, 0.0, 0.0), (0.0, 0.0, 50.0)),
    ("skewed", (50.0, 10.0, 0.0), (20.0, 45.0, 5.0)),
    ("mirrored", (-50.0, 0.0, 0.0), (0.0, 50.0, 0.0)),
    ("anisotropic", (90.0, 0.0, 0.0), (0.0, 11.0, 0.0))])
def test_nodes_on_any_slice(pkg, ctx, name, X, Y):
    A = [-0.5 * (x + y) + 0.7 for x, y in zip(X, Y)]
    rows = [((0.0, 0.0, 1.5), 4.0, 1.4 + 0.03j), ((12.0, -10.0, -2.0), 2.5, 1.6 + 0.0j),
            ((-15.0, 4.0, 6.0), 3.0, 1.3 + 0.2j)]
    check(both(pkg, ctx, quad(pkg, A, X, Y), 320, 300, 3.0, rows))


@pytest.mark.parametrize("count", [63, 64, 65, 130])
def test_nodes_of_many_spheres(pkg, ctx, count):
    """Tile masks of one, two and three words, orders of several buckets."""
    rng = np.random.default_rng(count)
    rows = [((float(x), float(y), float(z)), float(a), complex(1.4 + 0.1 * a, 0.01))
            for x, y, z, a in zip(rng.uniform(-60, 60, count), rng.uniform(-60, 60, count),
                                  rng.choice([0.0, 1.0], count), rng.uniform(0.3, 3.0, count))]
    q = quad(pkg, (-60.0, -60.0, 0.0), (120.0, 0.0, 0.0), (0.0, 120.0, 0.0))
    check(both(pkg, ctx, q, 384, 384, 4.0, rows, nk=16))


@pytest.mark.parametrize("case", ["tiny spheres", "one large sphere", "all outside", "coarse",
                                  "very fine", "high order"])
def test_nodes_at_the_ends_of_their_range(pkg, ctx, case):
    lam, L, N, rows = 3.0, 60.0, 320, ROWS
    if case == "tiny spheres":       # far sooner than their order's reach: the half-edge rule
        rows = [((float(x), 3.0 - x, 0.0), 0.05, 1.5 + 0.0j) for x in range(-12, 13, 2)]
    elif case == "one large sphere":   # every tile near it
        rows = [((0.0, 0.0, 0.0), 14.0, 1.5 + 0.05j)] * 2
    elif case == "all outside":
        rows = [((60.0 + 10.0 * i, 5.0 * i, 0.0), 4.0, 1.5 + 0.01j) for i in range(4)]
    elif case == "coarse":           # pixels near half a wavelength: no tile is worth it
        L = 400.0
    elif case == "very fine":        # the whole slice a wavelength
        L, rows = 3.0, [((5.0 * i, 9.0, 0.0), 4.0, 1.5 + 0.01j) for i in range(-2, 3)]
    else:
        lam, L, rows = 1.0, 30.0, [((0.0, 0.0, 0.0), 9.0, 1.2 + 0.01j),
                                   ((9.0, 11.0, 0.0), 3.0, 1.4 + 0.0j)]
    q = quad(pkg, (-L / 2, -L / 2, 0.0), (L, 0.0, 0.0), (0.0, L, 0.0))
    check(both(pkg, ctx, q, N, N, lam, rows))


def test_nodes_accumulate(pkg, ctx):
    q = quad(pkg, (-30.0, -30.0, 0.0), (60.0, 0.0, 0.0), (0.0, 60.0, 0.0))
    check(both(pkg, ctx, q, 300, 300, 3.0, ROWS, accumulate=True))


def test_node_batches_eager_captured_and_per_call(pkg, ctx):
    """Instances with nodes and without (small, no spheres) in one batch: the
    same images eagerly and replayed, with other work between the replays,
    and the per-call pipeline's, whose plans are small enough to keep to
    their pixels."""
    import bimsim_amd.pipeline as P
    import bimsim_amd.workloads as W
    insts = [W.config(2, N=512, nk=32), W.config(1, N=48, nk=32), W.config(2, N=512, nk=48),
             W.config(2, N=320, nk=24)]
    waves = [W.mc_waves(i, pkg.mc_sample_na) for i in insts]
    arr, spheres, Wv, n = P.batch_tables(insts, waves)
    wd = torch.as_tensor(Wv.ravel()).cuda()
    imgs = []
    for graph in (False, True):
        D, Di, Ab = (torch.zeros(n, dtype=torch.float32, device="cuda") for _ in range(3))
        b = ctx.batch(arr, spheres, wd, D, Di, Ab, prec=pkg.FP32_FAST, use_graph=graph)
        first = D.clone()
        for _ in range(3):
            D.fill_(3.0)
            P.simulate(ctx, insts[1], torch.as_tensor(waves[1]).cuda(), pkg.FP32_FAST)
            b.launch()
            torch.cuda.synchronize()
            assert torch.equal(D, first)
        imgs.append(first)
        b.close()
    assert torch.equal(imgs[0], imgs[1])
    off = 0
    for i, w in zip(insts, waves):
        one = P.simulate(ctx, i, torch.as_tensor(w).cuda(), pkg.FP32_FAST)
        m = i["Nd"] ** 2
        assert (imgs[0][off: off + m] - one.D).norm() <= 2e-6 * one.D.norm()
        off += m


def test_plans_with_and_without_nodes_are_tuned_apart(pkg, monkeypatch, capfd):
    """Two plans of one shape (pixels, spheres, orders, waves), the spheres over
    a narrow slice and a wide one: without nodes and with them, so that the
    kernel variant timed for one is not taken for the other; a third like the
    second takes its."""
    monkeypatch.setenv("BIMSIM_TUNE_LOG", "1")
    c = pkg.Context(0)
    k, N, tuned = 1.5, 512, []
    rng = np.random.default_rng(5)
    at = [(0.0, 0.0)] + [tuple(rng.uniform(-0.5, 0.5, 2)) for _ in range(9)]
    spheres, n = [], 0
    for i in range(10):
        a = 8.0 / k / (1.0 + 0.02 * i)
        spheres.append(dict(a=a, n=1.4 + 0.02j, coeff_off=n, Nl=pkg.sphere_order(a, 2 * math.pi / k)))
        n += spheres[-1]["Nl"] + 1
    A, B = (torch.zeros(n, dtype=torch.complex128, device="cuda") for _ in range(2))
    w = torch.tensor(pkg.mc_sample_na(32, (0.0, 0.0, 1.0), 0.1, 0.6, pkg.RNG_SPLITMIX64, 1),
                     dtype=torch.float64).cuda()
    U = torch.empty(N * N, dtype=torch.complex64, device="cuda")
    capfd.readouterr()
    for width in (20.0, 60.0, 60.01):
        for s, (x, y) in zip(spheres, at):
            s["p"] = (x * width, y * width, 0.0)
        c.mie_coeffs(spheres, k, A, B)
        c.nf_us(pkg.Quad.xy(width), N, N, (0.0, 0.0, 0.0), k, spheres, A, B, w, 1.0, U,
                prec=pkg.FP32_FAST)
        torch.cuda.synchronize()
        tuned.append(capfd.readouterr().err.count("harmonic waves per SIMD"))
    assert tuned == [1, 1, 0]
    c.close()
