"""Analytic multihit at its range edges: on a cold lattice the staple of every
temporal link is 6 xi, so the temporal link is I1(x) / I0(x) with x = 6 xi beta
-- each side of the polynomials' limits x = 6 and x = 12, the series beyond, and
small x -- against scipy's exponentially scaled Bessel functions.  Tolerance: the
Horner sums and the division are each good to a few units of 2^-53 and scipy's
functions to about as much: 16 units, 1.8e-15; beyond x = 12 the running sums'
error grows with the number of terms: 1e-14 as for the Bessel self test."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["F64", "F32"])
@pytest.mark.parametrize("x", [1e-4, 0.3, 3.0, 5.999999, 6.0, 6.000001, 9.0, 11.99999, 12.0, 12.00001, 20.0, 40.0])
def test_analytic_multihit_ratio(u1, prec, x):
    sp = pytest.importorskip("scipy.special")
    lat = u1.Lattice.cold(u1.geom((2, 2, 2, 2), x / 6.0, 1.0), getattr(u1, prec))
    t = lat.temporal_links(u1.POLY_MULTIHIT)
    beta_s = 6.0 * (x / 6.0)
    want = sp.ive(1, beta_s) / sp.ive(0, beta_s)
    assert np.all(t.imag == 0.0)
    assert np.max(np.abs(t.real / want - 1.0)) <= (1.8e-15 if x < 12.0 else 1e-14)


@pytest.mark.parametrize("nt", [2, 8, 10])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_polyakov_loads_in_groups(u1, orc, mode, nt):
    """The product and the sum along t take their loads in groups of eight:
    below, at and past one group, against the oracle."""
    dims = (4, 6, 2, nt)
    g, og = u1.geom(dims, 1.1, 1.2), orc.geom(dims, 1.1, 1.2)
    ref = orc.hotstart(og, 23)
    ref[::7] += 2 * np.pi  # angles outside [-pi, pi]: the general wrap
    lat = u1.Lattice.from_host(g, ref)
    c_gpu = lat.poly2(mode, u1.metro(1, 5, 3.0), 23)
    c_orc = orc.poly2(og, ref, mode, orc.metro(1, 5, 3.0), 23)
    assert np.allclose(c_gpu, c_orc, rtol=1e-12, atol=1e-15)
    assert abs(lat.polyakov() - orc.polyakov(og, ref)) <= 1e-14


@pytest.mark.parametrize("prec,tol", [("F64", 1e-12), ("F32", 1e-12)])
@pytest.mark.parametrize("dims", [(2, 2, 2, 2), (4, 6, 2, 16), (6, 2, 10, 18), (4, 4, 4, 32), (4, 4, 4, 34)])
def test_analytic_loops_are_the_products_of_the_links(u1, orc, prec, tol, dims):
    """Loops formed in one workgroup per 32 spatial sites (8, 48, 120 and 64 sites,
    one to 32 rows of time slices; 34: through the field) against the product of
    the links themselves, a chain of at most 34 complex products."""
    g, og = u1.geom(dims, 1.1, 1.2), orc.geom(dims, 1.1, 1.2)
    ref = orc.hotstart(og, 31)
    lat = u1.Lattice.from_host(g, ref)
    if prec == "F32":
        lat = lat.astype(u1.F32)
    links = lat.temporal_links(u1.POLY_MULTIHIT).reshape(dims[3], -1)
    P = lat.poly_volume(u1.POLY_MULTIHIT)
    assert np.allclose(P.reshape(-1), np.prod(links, axis=0), rtol=tol, atol=1e-15)
    if prec == "F64":
        assert np.allclose(P, orc.poly_volume(og, ref, 1), rtol=tol, atol=1e-15)
