"""Plaquette component fields (k_plaquette_fields) at the edges of its launch:
less than one workgroup, a remainder, extents that are no power of two, and more
sites than kFoldRows workgroups hold at once.  Against the oracle to 1e-13 (sines
and sums in another order, as in test_gpu_parity), binary32 input against the
same angles in binary64."""
import numpy as np
import pytest

from tests.test_gpu_parity import make_pair, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(2, 2, 2, 2), (6, 10, 4, 2), (14, 6, 10, 4), (32, 32, 32, 34)])
def test_plaquette_fields_edges(u1, orc, dims):
    g, og, lat, ref = make_pair(u1, orc, dims, 1.0, 1.0, True, seed=5)
    say(f"plaquette fields {dims}")
    no = lat.convert_layout(True)
    for st in (True, False):
        Fo, mo = orc.plaquette_fields(og, ref, st, True)
        for F, m in (lat.plaquette_fields(st, True), no.plaquette_fields(st, False)):
            assert np.max(np.abs(F - Fo)) <= 1e-13
            assert np.max(np.abs(m - mo)) <= 1e-13
    # binary32 angles: |error of P| <= 4 units of pi 2^-23, and as much again in the sum of four
    F32, _ = lat.astype(u1.F32).plaquette_fields(True, True)
    assert np.max(np.abs(F32 - orc.plaquette_fields(og, ref, True, True)[0])) <= 8 * np.pi * 2.0 ** -22
