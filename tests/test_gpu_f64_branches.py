"""Branches that the binary64 update kernels take by a vote of the wavefront -- the
special cases of the angle of the staple, the second steps of the wrap, the accept
test of couplings whose weights may leave the range of exp -- against the oracle,
bit for bit (a NaN: in the same places)."""
import numpy as np
import pytest

from tests.test_gpu_parity import bits, say

pytestmark = pytest.mark.gpu

DIMS = (8, 6, 4, 6)


def same(a, b):
    nan = np.isnan(b)
    return np.array_equal(np.isnan(a), nan) and np.array_equal(bits(a[~nan]), bits(b[~nan]))


# xi: weights xi and 1 / xi of the staples.  5e-324, 1e-323: zero, denormal and infinite
# components; 1e308: sums of the components that overflow, and infinite ones
@pytest.mark.parametrize("xi", [1.0, 1.3, 5e-324, 1e-323, 2e-308, 1e308])
@pytest.mark.parametrize("links", ["thermal", "wide", "few", "cold", "nan"])
def test_overrelaxation_branches(u1, orc, xi, links):
    rng = np.random.default_rng(17)
    n = 4 * int(np.prod(DIMS))
    th = {"thermal": rng.uniform(-np.pi, np.pi, n),
          "wide": rng.uniform(-40.0, 40.0, n),                                        # several turns off
          "few": np.where(rng.random(n) < 2.0 / 64, 20.0, 0.5) * rng.normal(size=n),  # a lane or two per wavefront
          "cold": rng.choice([0.0, -0.0, np.pi, -np.pi], n),
          "nan": np.where(rng.random(n) < 0.01, rng.choice([np.nan, np.inf, -np.inf], n), rng.normal(size=n))}[links]
    say(f"fp64 overrelaxation branches xi {xi} {links}")
    g, og = u1.geom(DIMS, 1.0, xi), orc.geom(DIMS, 1.0, xi)
    lat = u1.Lattice.from_host(g, th)
    ref = th.copy()
    for parity in range(2):
        for mu in range(4):
            lat.phase(1, parity, mu, u1.BENCH_METRO, 1)
            orc.overrelax_phase(og, ref, parity, mu)
            assert same(lat.to_host(), ref), (parity, mu)


# 12 beta xi up to 650: no vote (54.1 just below); beyond: weights up to e^(2 beta |S|),
# past both ends of exp's range for 1e4
@pytest.mark.parametrize("beta,xi", [(54.1, 1.0), (54.2, 1.0), (60.0, 1.0), (1e4, 1.0), (-300.0, 1.3), (40.0, 0.01)])
@pytest.mark.parametrize("proposal", [0, 1])
def test_accept_branches(u1, orc, beta, xi, proposal):
    say(f"fp64 accept test beta {beta} xi {xi} proposal {proposal}")
    g, og = u1.geom(DIMS, beta, xi), orc.geom(DIMS, beta, xi)
    m, om = u1.metro(proposal, 7, 0.3), orc.metro(proposal, 7, 0.3)
    lat = u1.Lattice.cold(g, u1.F64)
    lat.hotstart(23)
    ref = orc.hotstart(og, 23)
    for s in range(2):
        assert lat.update(1, 1, m, 23, s, count_accepts=True) == orc.update(og, ref, 1, 1, om, 23, s, count_accepts=True)
        assert np.array_equal(bits(lat.to_host()), bits(ref))
