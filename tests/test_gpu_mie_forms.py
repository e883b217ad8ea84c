"""The closed form of the Mie coefficients (spheres whose order belongs to
their size) and the general one, at the edges of either, against the oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def run(pkg, ctx, spheres, kmag, quirks):
    off = 0
    for s in spheres:
        s["p"], s["coeff_off"] = (0.0, 0.0, 0.0), off
        off += s["Nl"] + 1
    A = torch.full((off + 3,), 7.0, dtype=torch.complex128, device="cuda")
    B = A.clone()
    ctx.mie_coeffs(spheres, kmag, A, B, quirks=quirks)
    assert bool((A[off:] == 7.0).all()) and bool((B[off:] == 7.0).all())
    return A.cpu().numpy(), B.cpu().numpy()


# k a at the limits of the closed form (0.01; 12, above which y_0 takes the
# reference's defect) and on either side of them, small and large
XS = [0.009, 0.011, 0.3, 1.0, 4.0, 11.5, 11.999999, 12.0, 12.000001, 25.0, 63.0, 140.0]


@pytest.mark.parametrize("quirks", [1, 0])
@pytest.mark.parametrize("n", [1.5 + 0.0j, 1.2 + 0.3j, 1.7 + 1e-6j, 0.8 + 0.02j])
def test_coefficients_at_the_edges_of_the_closed_form(pkg, ctx, orc, n, quirks):
    kmag = 2.0
    spheres = [dict(a=x / kmag, n=n, Nl=pkg.sphere_order(x / kmag, 2 * np.pi / kmag)) for x in XS]
    got = run(pkg, ctx, spheres, kmag, quirks)
    for s in spheres:
        want = orc.mie_coeffs(s["Nl"], kmag, s["a"], n, quirks)
        sl = slice(s["coeff_off"], s["coeff_off"] + s["Nl"] + 1)
        for g, w in zip(got, want):
            # the oracle's power series (|z| <= 12) and recurrences lose up to
            # 5e-12; each of the twelve spheres is a call of one below
            assert np.linalg.norm(g[sl] - w) <= 1e-11 * np.linalg.norm(w), s
        one = run(pkg, ctx, [dict(s)], kmag, quirks)
        for g, w in zip(one, want):
            assert np.linalg.norm(g[: s["Nl"] + 1] - w) <= 1e-11 * np.linalg.norm(w), s


@pytest.mark.parametrize("count", [1, 7, 8, 9, 63, 64, 65, 130])
def test_coefficients_of_many_spheres(pkg, ctx, orc, count):
    """Partial blocks and launches of the closed form, orders mixed."""
    kmag = 1.3
    spheres = [dict(a=0.2 + 0.37 * (i % 23), n=complex(1.3 + 0.01 * (i % 20), 0.004 * (i % 9)))
               for i in range(count)]
    for s in spheres:
        s["Nl"] = pkg.sphere_order(s["a"], 2 * np.pi / kmag)
    A, B = run(pkg, ctx, spheres, kmag, 1)
    for s in spheres:
        sl = slice(s["coeff_off"], s["coeff_off"] + s["Nl"] + 1)
        a, b = orc.mie_coeffs(s["Nl"], kmag, s["a"], s["n"], 1)
        assert np.linalg.norm(A[sl] - a) <= 1e-11 * np.linalg.norm(a), s
        assert np.linalg.norm(B[sl] - b) <= 1e-11 * np.linalg.norm(b), s


@pytest.mark.parametrize("extra", [19, 21, 40])
def test_orders_past_the_closed_form(pkg, ctx, orc, extra):
    """A sphere with more orders than its size asks for: up to 20 past x + 4
    x^(1/3) the closed form, beyond it the general one for the whole call."""
    kmag, a, n = 2.0, 3.0, 1.4 + 0.05j
    x = kmag * a
    spheres = [dict(a=a, n=n, Nl=int(x + 4.05 * x ** (1 / 3)) + extra),
               dict(a=1.0, n=n, Nl=9)]
    A, B = run(pkg, ctx, spheres, kmag, 1)
    for s in spheres:
        sl = slice(s["coeff_off"], s["coeff_off"] + s["Nl"] + 1)
        a_, b_ = orc.mie_coeffs(s["Nl"], kmag, s["a"], n, 1)
        assert np.linalg.norm(A[sl] - a_) <= 1e-11 * np.linalg.norm(a_), s
        assert np.linalg.norm(B[sl] - b_) <= 1e-11 * np.linalg.norm(b_), s


# k a and an index far below one, whose orders run past |n| k a by far: on both
# sides of where the closed form's recurrence would leave its range, and past
# where it would overflow (x = 160, 360 and 800 for these indices)
@pytest.mark.parametrize("x,n", [(60.0, 0.01), (120.0, 0.01), (160.0, 0.01), (150.0, 0.1),
                                 (160.0, 0.1), (400.0, 0.1), (350.0, 0.3), (800.0, 0.3)])
def test_index_far_below_one(pkg, ctx, orc, x, n):
    kmag = 2.0
    s = dict(a=x / kmag, n=complex(n), Nl=pkg.sphere_order(x / kmag, 2 * np.pi / kmag))
    A, B = run(pkg, ctx, [s], kmag, 1)
    a, b = orc.mie_coeffs(s["Nl"], kmag, s["a"], s["n"], 1)
    # (the reference's own arrays leave the range at the highest orders)
    there = np.isfinite(a) & np.isfinite(b)
    assert there.sum() > 0.5 * len(a)
    A, B = (g[: s["Nl"] + 1][there] for g in (A, B))
    a, b = a[there], b[there]
    assert np.linalg.norm(B - b) <= 1e-11 * np.linalg.norm(b)
    # A grows over the orders by up to 1e200: each order by itself
    assert (np.abs(A - a) <= 1e-9 * np.abs(a)).all()
