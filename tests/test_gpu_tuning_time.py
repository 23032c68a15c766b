"""Tuning where walks are hopeless: with gcd(Nz, Nt) = 2 diagonals a walk takes up to
fifteen times as long as the two phases.  Timing every shape of them over and over
made the first call nine times as long as tuning the phases alone; one look at each
about doubles it."""
import time

import pytest

from tests.test_gpu_parity import say

pytestmark = pytest.mark.gpu


def test_first_call_with_few_diagonals(u1):
    t = {}
    # (the same planes; entries are kept per extents.  Warmed up by a small lattice.)
    for pairs, dims in ((1, (4, 4, 6, 2)), (0, (20, 28, 36, 22)), (1, (28, 20, 36, 22))):
        u1.set_pair_fusion(pairs)
        try:
            lat = u1.Lattice.cold(u1.geom(dims, 1.0), u1.F64)
            lat.hotstart(3)
            u1.sync()
            t0 = time.perf_counter()
            lat.update(1, 3, u1.BENCH_METRO, 3, 0)
            u1.sync()
            t[pairs] = time.perf_counter() - t0
        finally:
            u1.set_pair_fusion(1)
    say(f"first call {1e3 * t[0]:.0f} ms without pairs and walks, {1e3 * t[1]:.0f} ms with")
    assert t[1] < 5 * t[0]
