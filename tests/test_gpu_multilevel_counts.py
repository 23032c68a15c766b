"""Pass counts that u1_multilevel refuses, and calls without sublattice updates, which
never look at them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("metrop,ovrn", [(-1, 3), (1, -3), (4096, 0)])
def test_bad_pass_counts(u1, metrop, ovrn):
    lat = u1.Lattice.cold(u1.geom((4, 4, 4, 8), 1.0), u1.F64)
    lat.hotstart(3)
    for k4, k2 in ((0, 1), (1, 0), (1, 1)):
        with pytest.raises(u1.U1Error, match="U1_ERR_ARG: bad pass counts"):
            lat.multilevel(1, k4, 1, k2, metrop, ovrn, u1.BENCH_METRO, 5)
    assert np.array_equal(lat.multilevel(1, 0, 1, 0, metrop, ovrn, u1.BENCH_METRO, 5),
                          lat.multilevel(1, 0, 1, 0, 1, 1, u1.BENCH_METRO, 5))
