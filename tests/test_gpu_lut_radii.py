"""The radial tables' own recurrences (orders that belong to the size) and the
general form at the edges of either, against the oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# k a = 2 a; orders at and past the limit k lo + 4.05 cbrt + 20; distances
# from the sphere's edge and from beyond it; small arguments of many orders,
# whose unscaled values leave the range of a double; real and absorbing n
@pytest.mark.parametrize("a,n,over,dmin,dmax,dR,aR", [
    (0.006, 1.4 + 0.1j, 0, 0.0, 3.0, 65, 5), (0.5, 1.3 + 0.0j, 0, 0.0, 40.0, 130, 2),
    (3.0, 1.5 + 0.2j, 0, 0.5, 20.0, 64, 300), (3.0, 1.5 + 0.2j, 16, 0.5, 20.0, 63, 64),
    (3.0, 1.5 + 0.2j, 30, 0.5, 20.0, 33, 65), (3.0, 0.7 + 0.0j, 3, 9.0, 30.0, 2, 129),
    (12.0, 1.45 + 0.01j, 0, 0.0, 60.0, 257, 2048), (40.0, 1.2 + 0.5j, 5, 1.0, 90.0, 100, 1500)])
def test_radial_tables(pkg, ctx, orc, a, n, over, dmin, dmax, dR, aR):
    kmag = 2.0
    nl = pkg.sphere_order(a, 2 * np.pi / kmag) + over
    s = dict(p=(0.0, 0.0, 0.0), a=a, n=n, Nl=nl, coeff_off=0)
    h = torch.empty(dR * (nl + 1), dtype=torch.complex128, device="cuda")
    j = torch.empty(aR * (nl + 1), dtype=torch.complex128, device="cuda")
    ctx.sphere_radial_lut(s, kmag, dmin, dmax, dR, aR, h, j)
    want_h = orc.lut_hankel(nl, kmag, a, dmin, dmax, dR)
    want_j = orc.lut_bessel(nl, kmag, a, n, aR)
    got_h, got_j = h.cpu().numpy().reshape(dR, nl + 1), j.cpu().numpy().reshape(aR, nl + 1)
    def close(got, want):
        # per order: the functions span many powers of ten.  The oracle's power
        # series and recurrences lose up to 5e-12 of an order's largest value
        top = np.abs(want).max(axis=0)
        assert (np.abs(got - want).max(axis=0) <= 1e-11 * top + 1e-200).all()

    for got, want in ((got_h.real, want_h.real), (got_h.imag, want_h.imag), (got_j, want_j)):
        close(got, want)
    # either table alone, which may take the other form than both together: each
    # value written, and to the same bound
    h2, j2 = torch.full_like(h, np.nan), torch.full_like(j, np.nan)
    ctx.sphere_radial_lut(s, kmag, dmin, dmax, dR, 0, h2, None)
    ctx.sphere_radial_lut(s, kmag, dmin, dmax, 0, aR, None, j2)
    one_h, one_j = h2.cpu().numpy().reshape(got_h.shape), j2.cpu().numpy().reshape(got_j.shape)
    for one, both in ((one_h.real, got_h.real), (one_h.imag, got_h.imag), (one_j, got_j)):
        close(one, both)
