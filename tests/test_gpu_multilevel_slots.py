"""Multilevel accumulation in more than one chunk of product slots (256 MiB of them: 32
level-2 steps at 32^4), with products that differ from step to step: stochastic
multihit links of level-2 step c = i n2 + k, which u1_temporal_links gives for
Philox word c, summed here step by step.  A slot read twice, late or not at all
changes the field by about the links' spread (0.1) over the steps.  Steps, level
products and the eight layer pairs: 33 * 2 * 8 additions and products of 2^-53 and
as many again here, 1.2e-13 relative."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_chunked_steps(u1):
    n, n4, n2, seed, call = 32, 2, 33, 5, 2
    lat = u1.Lattice.cold(u1.geom((n, n, n, n), 1.0), u1.F32)
    mh = u1.metro(u1.PROPOSAL_DELTA, 2, 0.1)
    _, field = lat.multilevel(n4, 0, n2, 0, 1, 1, u1.BENCH_METRO, seed, call, u1.POLY_MULTIHIT_STOCHASTIC, mh, field=True)
    field = field.reshape(3, n // 2, n, n, n)  # dir, R - 1, z, y, x
    level4 = {}
    for i in range(n4):
        level2 = {}
        for k in range(n2):
            t = lat.temporal_links(u1.POLY_MULTIHIT_STOCHASTIC, mh, seed, u1.STREAM_ML_MULTIHIT, i * n2 + k, call)
            t = t.reshape(n // 2, 2, n, n, n)
            p = t[:, 0] * t[:, 1]
            for d, r in ((0, 1), (1, 16), (2, 7)):
                level2[d, r] = level2.get((d, r), 0.0) + p * np.roll(p, -r, axis=3 - d).conj()
        for key, s in level2.items():
            s = (s / n2).reshape(n // 4, 2, n, n, n)
            level4[key] = level4.get(key, 0.0) + s[:, 0] * s[:, 1]
    for (d, r), s in level4.items():
        want = np.prod(s / n4, axis=0)
        assert np.max(np.abs(field[d, r - 1] / want - 1.0)) <= 1.2e-13, (d, r)
