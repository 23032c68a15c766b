"""Fused pairs that take several steps over a plane (k_pair): one step between
phase 0 and phase 1 where a step covers two rows, phase by phase where it does
not.  Shapes forced through the tune cache; binary64 bit for bit against the
oracle with identical accept counts, binary32 bit for bit against separate
launches, plaquettes to summation order (1e-13, 1e-12)."""
import numpy as np
import pytest

from tests.test_gpu_parity import bits, make_pair, say

pytestmark = pytest.mark.gpu

# dims, block, sites per thread: planes of Nx Ny / 2 sites, rows of Nx / 2
SHAPES = [
    ((64, 6, 2, 4), 64, 1),     # a step is exactly two rows: 3 steps
    ((12, 22, 4, 2), 64, 1),    # 132 = 2 * 64 + 4 sites: the last step one row less
    ((10, 26, 2, 4), 128, 1),   # 130 = 128 + 2: less than a row left for the second step
    ((24, 48, 2, 4), 64, 1),    # 576 = 9 * 64: an odd number of steps
    ((16, 32, 2, 4), 128, 1),   # 256 = 2 * 128
    ((72, 8, 2, 4), 64, 1),     # a step is less than two rows: phase by phase
    ((24, 20, 2, 4), 64, 2),    # two sites per thread: phase by phase
]


@pytest.fixture
def forced(u1, tmp_path):
    def force(dims, block, spt, suffix):
        vol = "x".join(map(str, dims))
        rows = [f"{vol}\t{k}{name}_{suffix}\tthreads=halfvolume\t{b}\t{s}\t{z}\t0\t1\t1\t0\t# forced"
                for k in ("Metropolis", "OverRelaxation")
                for name, b, s, z in (("", 64, 1, 1), ("Pair", block, spt, 2), ("Walk", 0, 1, 1))]
        p = tmp_path / "pair.csv"
        p.write_text("tunecache\tlatticeu1_amd-1\tgpu_arch=gfx950\nvolume\tname\taux\n" + "\n".join(rows) + "\n")
        u1.tune_load(str(p))

    u1.tune_enable(False)
    u1.set_pass_fusion(0)
    yield force
    u1.set_pair_fusion(1)
    u1.set_pass_fusion(1)
    u1.tune_enable(True)


@pytest.mark.parametrize("dims,block,spt", SHAPES)
def test_fp64_pair_steps_parity(u1, orc, forced, dims, block, spt):
    forced(dims, block, spt, "f64")
    g, og, lat, ref = make_pair(u1, orc, dims, 0.9, 1.3, True, seed=53)
    say(f"fp64 pair steps {dims} {block} x {spt}")
    m, om = u1.BENCH_METRO, orc.metro(1, 4, 0.5)
    for s, ml in ((0, 0), (1, 2), (2, 4)):
        assert lat.update(1, 2, m, 53, s, mask_ml=ml, count_accepts=True) == \
            orc.update(og, ref, 1, 2, om, 53, s, mask_ml=ml, count_accepts=True)
        assert np.array_equal(bits(lat.to_host()), bits(ref)), s
    p = lat.update_plaquette(1, 1, m, 53, 3)
    orc.update(og, ref, 1, 1, om, 53, 3)
    assert np.array_equal(bits(lat.to_host()), bits(ref))
    assert np.max(np.abs(p - orc.plaquette(og, ref))) <= 1e-13


@pytest.mark.parametrize("dims,block,spt", SHAPES + [((96, 96, 2, 4), 256, 1)])
def test_fp32_pair_steps_match_separate(u1, forced, dims, block, spt):
    forced(dims, block, spt, "f32")
    g = u1.geom(dims, 1.0, 1.0)
    out = {}
    for mode in (0, 1):
        u1.set_pair_fusion(mode)
        lat = u1.Lattice.cold(g, u1.F32)
        lat.hotstart(29)
        acc = [lat.update(1, 2, u1.BENCH_METRO, 29, s, mask_ml=ml, count_accepts=True)
               for s, ml in ((0, 0), (1, 2), (2, 4))]
        p = lat.update_plaquette(1, 2, u1.BENCH_METRO, 29, 3)
        out[mode] = (lat.to_host(), acc, p)
    say(f"fp32 pair steps {dims} {block} x {spt}: accepts {out[1][1]}")
    assert np.array_equal(out[0][0], out[1][0])
    assert out[0][1] == out[1][1]
    assert np.max(np.abs(out[0][2] - out[1][2])) <= 1e-12
