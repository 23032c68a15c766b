"""One-launch sweeps whose workgroups do not find each other: with no patience for
the others to begin, one workgroup does the whole sweep (of its slab).  Binary64
bit for bit against the oracle, binary32 against a launch per phase, identical
accept counts; the plaquette to summation order.  Launches follow each other, so
that control words left behind by one would show in the next."""
import time

import numpy as np
import pytest

from tests.test_gpu_parity import bits, make_pair, say

pytestmark = pytest.mark.gpu

ALONE = 1  # flag of u1_selftest_sweep
# dims, workgroup size
SHAPES = [((2, 2, 2, 2), 64), ((4, 6, 10, 2), 64), ((8, 8, 8, 8), 64), ((8, 8, 8, 8), 512), ((12, 12, 20, 10), 256)]
PASSES = [(1, 3), (2, 0), (0, 1)]
MASKED = [((4, 6, 10, 6), 64, 4), ((8, 8, 8, 24), 128, 2), ((4, 4, 4, 512), 64, 2)]


@pytest.mark.parametrize("dims,block,ml", [(d, b, 0) for d, b in SHAPES] + MASKED)
def test_fp64_alone_parity(u1, orc, dims, block, ml):
    g, og, lat, ref = make_pair(u1, orc, dims, 0.9, 1.3, True, seed=67)
    say(f"fp64 one-launch sweep by one workgroup {dims} {block} mask {ml}")
    m, om = u1.metro(1, 3, 0.5), orc.metro(1, 3, 0.5)
    for s, flags in enumerate((ALONE, 0, ALONE)):
        a, b = PASSES[s]
        got = u1.selftest_sweep(lat, a, b, m, 67, s, block, flags, mask_ml=ml)
        assert got == orc.update(og, ref, a, b, om, 67, s, mask_ml=ml, count_accepts=True), s
        assert np.array_equal(bits(lat.to_host()), bits(ref)), s
    if ml == 0:
        for s, (a, b) in enumerate(PASSES):
            acc, p = u1.selftest_sweep(lat, a, b, m, 67, 8 + s, block, ALONE, plaquette=True)
            assert acc == orc.update(og, ref, a, b, om, 67, 8 + s, count_accepts=True)
            assert np.array_equal(bits(lat.to_host()), bits(ref)), s
            assert np.max(np.abs(p - orc.plaquette(og, ref))) <= 1e-13


@pytest.mark.parametrize("dims,block,ml", [(d, b, 0) for d, b in SHAPES] + MASKED + [((16, 16, 16, 8), 1024, 0)])
def test_fp32_alone_matches_phases(u1, dims, block, ml):
    g = u1.geom(dims, 1.0, 1.2)
    say(f"fp32 one-launch sweep by one workgroup {dims} {block} mask {ml}")
    one, ref = u1.Lattice.cold(g, u1.F32), u1.Lattice.cold(g, u1.F32)
    for lat in (one, ref):
        lat.hotstart(31)
    u1.tune_enable(False)
    u1.set_pass_fusion(0)  # a launch per phase
    try:
        for s, (a, b) in enumerate(PASSES):
            got = u1.selftest_sweep(one, a, b, u1.BENCH_METRO, 31, s, block, ALONE, mask_ml=ml)
            assert got == ref.update(a, b, u1.BENCH_METRO, 31, s, mask_ml=ml, count_accepts=True), s
            assert np.array_equal(one.to_host(), ref.to_host()), s
    finally:
        u1.set_pass_fusion(1)
        u1.tune_enable(True)


def test_selftest_sweep_arguments(u1):
    lat = u1.Lattice.cold(u1.geom((4, 4, 4, 4), 1.0), u1.F64)
    big = u1.Lattice.cold(u1.geom((16, 16, 16, 16), 1.0), u1.F64)
    for bad in (lambda: u1.selftest_sweep(lat, 0, 0, u1.BENCH_METRO, 1, 0, 64),
                lambda: u1.selftest_sweep(lat, 1, 1, u1.BENCH_METRO, 1, 0, 1024),
                lambda: u1.selftest_sweep(lat, 1, 1, u1.BENCH_METRO, 1, 0, 96),
                lambda: u1.selftest_sweep(lat, 1, 1, u1.BENCH_METRO, 1, 0, 64, 64),
                lambda: u1.selftest_sweep(lat, 1, 1, u1.BENCH_METRO, 1, 0, 64, mask_ml=2, plaquette=True),
                lambda: u1.selftest_sweep(lat, 1, 8192, u1.BENCH_METRO, 1, 0, 64),
                lambda: u1.selftest_sweep(big, 1, 1, u1.BENCH_METRO, 1, 0, 64)):
        with pytest.raises(u1.U1Error, match="U1_ERR_ARG"):
            bad()


def test_accepts_of_long_sweeps(u1):
    """More accepted hits per wavefront and sweep than 32 bits hold: 32 workgroups of one
    wavefront, 512 sites a phase each, 129 passes of 8190 hits are 4.33e9.  At beta = 0 a
    binary32 hit is refused for accept words that round to 2^32 only, one in 2^25."""
    dims = (16, 16, 16, 8)
    lat = u1.Lattice.cold(u1.geom(dims, 0.0), u1.F32)
    hits = 4 * int(np.prod(dims)) * 129 * 8190
    say(f"fp32 one-launch sweep of 129 passes of 8190 hits {dims}")
    got = u1.selftest_sweep(lat, 129, 0, u1.metro(1, 8190, 0.5), 73, 0, 64)
    assert abs(got / hits - (1.0 - 2.0**-25)) < 1e-8


def test_tuning_time_of_long_sweeps(u1):
    """Choosing the launches of a sweep does not run that sweep over and over: the first
    call, tuning included, within ten of the second."""
    lat = u1.Lattice.cold(u1.geom((4, 4, 6, 4), 1.0), u1.F64)
    lat.hotstart(3)
    t = []
    for s in range(2):
        u1.sync()
        t0 = time.perf_counter()
        lat.update(0, 8000, u1.BENCH_METRO, 3, s)
        u1.sync()
        t.append(time.perf_counter() - t0)
    say(f"fp64 8000 passes: {t[0]:.3f} s with tuning, {t[1]:.3f} s without")
    assert t[0] < 10 * t[1]
