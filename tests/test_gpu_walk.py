"""The (parity, 2) + (parity, 3) walk (k_walk): shapes forced through the tune
cache, at the edges of its dispatch -- one wavefront and many, segments of one
step, uneven last segments, strips past the end of a plane, Nz != Nt, every
order, multilevel masks.  FP64 bit for bit against the oracle with identical
accept counts; FP32, which has no oracle, bit for bit against the separate
phases.  The in-sweep plaquette differs from the oracle's by summation order
only (1e-13, as for the other launch forms)."""
import numpy as np
import pytest

from tests.test_gpu_parity import bits, make_pair, say

pytestmark = pytest.mark.gpu

# dims, wavefronts, segments per wavefront, block.z (1: plain, 2 + 2 log2 strip groups)
SHAPES = [
    ((2, 2, 2, 2), 1, 1, 1),       # two planes per diagonal, every neighbour wraps
    ((6, 10, 4, 12), 5, 1, 2),     # Nz != Nt, last segment shorter
    ((8, 8, 8, 8), 2, 4, 4),       # one step per segment, half-empty strips
    ((18, 10, 6, 4), 3, 2, 8),     # P = 90: strips past the plane's end, uneven groups
    ((16, 12, 16, 8), 8, 1, 6),    # several strips, eight wavefronts
]


@pytest.fixture
def forced(u1, tmp_path):
    def force(dims, waves, segs, order, suffix):
        vol = "x".join(map(str, dims))
        rows = [f"{vol}\t{k}{name}_{suffix}\tthreads=halfvolume\t{b}\t{s}\t{z}\t0\t1\t1\t0\t# forced"
                for k in ("Metropolis", "OverRelaxation")
                for name, b, s, z in (("", 64, 1, 1), ("Pair", 0, 1, 1), ("Walk", 64 * waves, segs, order))]
        p = tmp_path / "walk.csv"
        p.write_text("tunecache\tlatticeu1_amd-1\tgpu_arch=gfx950\nvolume\tname\taux\n" + "\n".join(rows) + "\n")
        u1.tune_load(str(p))

    u1.tune_enable(False)
    u1.set_pass_fusion(0)
    yield force
    u1.set_pair_fusion(1)
    u1.set_pass_fusion(1)
    u1.tune_enable(True)


@pytest.mark.parametrize("dims,waves,segs,order", SHAPES)
def test_fp64_walk_parity(u1, orc, forced, dims, waves, segs, order):
    forced(dims, waves, segs, order, "f64")
    g, og, lat, ref = make_pair(u1, orc, dims, 0.9, 1.3, True, seed=71)
    say(f"fp64 walk parity {dims} {waves} wavefronts x {segs} segments, order {order}")
    m, om = u1.BENCH_METRO, orc.metro(1, 4, 0.5)
    for s in range(3):
        assert lat.update(1, 2, m, 71, s, count_accepts=True) == orc.update(og, ref, 1, 2, om, 71, s,
                                                                            count_accepts=True)
        assert np.array_equal(bits(lat.to_host()), bits(ref)), s
    for ml in (2, 4):
        assert lat.update(1, 1, m, 71, 3, mask_ml=ml, count_accepts=True) == \
            orc.update(og, ref, 1, 1, om, 71, 3, mask_ml=ml, count_accepts=True)
        assert np.array_equal(bits(lat.to_host()), bits(ref)), ml
    p = lat.update_plaquette(1, 1, m, 71, 4)
    orc.update(og, ref, 1, 1, om, 71, 4)
    assert np.array_equal(bits(lat.to_host()), bits(ref))
    assert np.max(np.abs(p - orc.plaquette(og, ref))) <= 1e-13


@pytest.mark.parametrize("dims,waves,segs,order", SHAPES + [((28, 20, 12, 22), 16, 1, 4), ((48, 48, 16, 16), 4, 2, 6)])
def test_fp32_walk_matches_phases(u1, forced, dims, waves, segs, order):
    forced(dims, waves, segs, order, "f32")
    g = u1.geom(dims, 1.0, 1.0)
    out = {}
    for mode in (0, 1):
        u1.set_pair_fusion(mode)
        lat = u1.Lattice.cold(g, u1.F32)
        lat.hotstart(19)
        acc = [lat.update(1, 2, u1.BENCH_METRO, 19, s, mask_ml=ml, count_accepts=True)
               for s, ml in ((0, 0), (1, 2), (2, 4))]
        p = lat.update_plaquette(1, 2, u1.BENCH_METRO, 19, 3)
        out[mode] = (lat.to_host(), acc, p)
    say(f"fp32 walk vs phases {dims} {waves} wavefronts x {segs} segments, order {order}: accepts {out[1][1]}")
    assert np.array_equal(out[0][0], out[1][0])
    assert out[0][1] == out[1][1]
    assert np.max(np.abs(out[0][2] - out[1][2])) <= 1e-12
