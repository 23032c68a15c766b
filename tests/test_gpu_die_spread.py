"""One-launch sweeps whose workgroups lie on several XCDs (dealt to them in turn, as
neighbours of a launch are): stores and counters at device scope instead of in one
L2.  Binary64 bit for bit against the oracle, binary32 against a launch per phase,
identical accept counts; the plaquette to summation order."""
import numpy as np
import pytest

from tests.test_gpu_parity import bits, make_pair, say

pytestmark = pytest.mark.gpu

ALONE, SPREAD = 1, 2  # flags of u1_selftest_sweep
PASSES = [(1, 3), (2, 0), (0, 1)]
# dims, workgroup size, mask: 32 workgroups on 8 XCDs, 15 and 4; slabs of 4, 16 and 1 workgroups
SHAPES = [((8, 8, 8, 8), 64, 0), ((4, 6, 10, 8), 64, 0), ((8, 8, 8, 8), 512, 0), ((8, 8, 8, 8), 128, 2),
          ((8, 8, 8, 24), 64, 4), ((4, 4, 4, 512), 64, 2)]


@pytest.mark.parametrize("dims,block,ml", SHAPES)
def test_fp64_spread_parity(u1, orc, dims, block, ml):
    g, og, lat, ref = make_pair(u1, orc, dims, 0.9, 1.3, True, seed=71)
    say(f"fp64 one-launch sweep over several XCDs {dims} {block} mask {ml}")
    m, om = u1.metro(1, 3, 0.5), orc.metro(1, 3, 0.5)
    for s, flags in enumerate((SPREAD, 0, SPREAD, SPREAD | ALONE, SPREAD)):
        a, b = PASSES[s % 3]
        got = u1.selftest_sweep(lat, a, b, m, 71, s, block, flags, mask_ml=ml)
        assert got == orc.update(og, ref, a, b, om, 71, s, mask_ml=ml, count_accepts=True), s
        assert np.array_equal(bits(lat.to_host()), bits(ref)), s
    if ml == 0:
        acc, p = u1.selftest_sweep(lat, 1, 3, m, 71, 9, block, SPREAD, plaquette=True)
        assert acc == orc.update(og, ref, 1, 3, om, 71, 9, count_accepts=True)
        assert np.max(np.abs(p - orc.plaquette(og, ref))) <= 1e-13


@pytest.mark.parametrize("dims,block,ml", SHAPES + [((16, 16, 16, 8), 1024, 0)])
def test_fp32_spread_matches_phases(u1, dims, block, ml):
    g = u1.geom(dims, 1.0, 1.2)
    say(f"fp32 one-launch sweep over several XCDs {dims} {block} mask {ml}")
    one, ref = u1.Lattice.cold(g, u1.F32), u1.Lattice.cold(g, u1.F32)
    for lat in (one, ref):
        lat.hotstart(37)
    u1.tune_enable(False)
    u1.set_pass_fusion(0)  # a launch per phase
    try:
        for s, (a, b) in enumerate(PASSES):
            got = u1.selftest_sweep(one, a, b, u1.BENCH_METRO, 37, s, block, SPREAD, mask_ml=ml)
            assert got == ref.update(a, b, u1.BENCH_METRO, 37, s, mask_ml=ml, count_accepts=True), s
            assert np.array_equal(one.to_host(), ref.to_host()), s
    finally:
        u1.set_pass_fusion(1)
        u1.tune_enable(True)
