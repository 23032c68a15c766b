"""Multilevel accumulation when the level-2 steps of a level-4 step need more
than one chunk of product slots (256 MiB of them: 32 steps at 32^4): one full
chunk, a chunk and a step, two chunks and a step.  Without sublattice updates
every step contributes the same products, so the per-site field equals that of
one step: n additions and one division by n are good to n units of 2^-53
relative per layer pair, eight layer pairs multiplied: 65 * 2 * 8 * 1.2e-16 =
1.3e-13."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n2", [32, 33, 65])
def test_chunks_match_one_step(u1, n2):
    lat = u1.Lattice.cold(u1.geom((32, 32, 32, 32), 1.0), u1.F32)
    lat.hotstart(5)
    want, f_want = lat.multilevel(1, 0, 1, 0, 1, 1, u1.BENCH_METRO, 3, field=True)
    got, f_got = lat.multilevel(2, 0, n2, 0, 1, 1, u1.BENCH_METRO, 3, field=True)
    big = np.abs(f_want) > 0
    assert np.max(np.abs(f_got[big] / f_want[big] - 1.0)) <= 1.3e-13
    assert np.allclose(got, want, rtol=0, atol=1.3e-13 * np.mean(np.abs(f_want)))
