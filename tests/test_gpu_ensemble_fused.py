"""Batched replicas with every fused launch forced (packed pairs, or pairs in
steps where a plane exceeds a workgroup, and walks), measuring sweeps included,
against no fusion: lattices bit for bit, plaquettes to summation order (1e-13,
as for the other launch forms)."""
import numpy as np
import pytest

from tests.test_gpu_parity import say

pytestmark = pytest.mark.gpu

# Nx Ny / 2 = 2, 18, 64 (one wavefront exactly), 72, 320 (the largest plane sets the block); Nz = Nt and not
PACKED = [(2, 2, 2, 2), (6, 6, 4, 10), (16, 8, 6, 4), (12, 12, 4, 8), (32, 20, 2, 6)]
# a plane of 1200 sites exceeds one workgroup in either precision: pairs in steps for all
STEPS = [(60, 40, 2, 4), (8, 8, 4, 4)]


@pytest.mark.parametrize("dims", [PACKED, STEPS], ids=["packed", "steps"])
@pytest.mark.parametrize("prec,ovrn", [("F32", 2), ("F64", 2), ("F64", 0)])
def test_ensemble_fused_matches_separate(u1, dims, prec, ovrn):
    geoms = [u1.geom(d, 1.0, 1.0 + 0.2 * i) for i, d in enumerate(dims)]
    out = {}
    try:
        u1.tune_enable(False)
        for mode in (0, 2):
            u1.set_pair_fusion(mode)
            e = u1.Ensemble(geoms, [91 + i for i in range(len(dims))], [1] * len(dims), getattr(u1, prec), 1, ovrn,
                            u1.BENCH_METRO)
            say(f"ensemble {prec} {dims} fusion mode {mode}, {ovrn} overrelaxation passes")
            e.sweep(2, graph=True)
            series = e.sweep_plaquette(3)
            out[mode] = ([e.read(r) for r in range(len(dims))], np.array(series))
            e.destroy()
    finally:
        u1.set_pair_fusion(1)
        u1.tune_enable(True)
    for r in range(len(dims)):
        assert np.array_equal(out[0][0][r], out[2][0][r]), dims[r]
    assert np.max(np.abs(out[0][1] - out[2][1])) <= 1e-13
