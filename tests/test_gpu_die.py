"""One-launch sweeps (k_die): all passes of a small lattice in one launch, forced
through the tune cache.  Binary64 bit for bit against the oracle with identical
accept counts, binary32 bit for bit against a launch per phase, plaquettes to
summation order (1e-13, 1e-12)."""
import numpy as np
import pytest

from tests.test_gpu_parity import bits, make_pair, say

pytestmark = pytest.mark.gpu

# dims, workgroup size
SHAPES = [
    ((2, 2, 2, 2), 64),      # 8 sites per phase: one workgroup, part of a wavefront
    ((4, 6, 10, 2), 64),     # 240 sites: the last of four wavefronts is partial
    ((4, 6, 10, 2), 512),    # one workgroup, half of its wavefronts without sites
    ((8, 8, 8, 8), 64),      # 32 workgroups of one wavefront
    ((8, 8, 8, 8), 256),     # 8 workgroups
    ((6, 10, 14, 6), 64),    # 2520 sites: 2 rounds, the second 7 wavefronts and a bit
    ((12, 12, 12, 10), 512), # 8640 sites: 17 workgroups, one round
    ((12, 12, 20, 10), 64),  # 14400 sites: 8 rounds, the last one wavefront
]
PASSES = [(1, 3), (2, 0), (0, 1)]
# dims, workgroup size, multilevel mask: every slab between frozen slices by itself
MASKED = [
    ((2, 2, 2, 2), 64, 2),      # one slab of 2 + 1 slices
    ((4, 6, 10, 6), 64, 4),     # slabs of four and two slices
    ((8, 8, 8, 24), 128, 2),    # 12 slabs: two on four of the XCDs
    ((6, 6, 6, 72), 64, 2),     # 36 slabs, 5 rows: 6 workgroups per slab
    ((12, 10, 8, 16), 64, 4),   # 1440 and 1920 sites on 16 workgroups: two rounds
    ((12, 10, 8, 16), 512, 2),
    ((4, 4, 4, 512), 64, 2),    # 256 slabs, 32 on an XCD: one workgroup each
]


@pytest.fixture
def forced(u1, tmp_path):
    def force(dims, block, suffix):
        vol = "x".join(map(str, dims))
        rows = [f"{vol}\tSweep{a}+{b}{mask}_{suffix}\tthreads=halfvolume\t{block}\t1\t1\t0\t1\t1\t0\t# forced"
                for a, b in PASSES for mask in ("", "Mask2", "Mask4")]
        p = tmp_path / "die.csv"
        p.write_text("tunecache\tlatticeu1_amd-1\tgpu_arch=gfx950\nvolume\tname\taux\n" + "\n".join(rows) + "\n")
        u1.tune_load(str(p))

    u1.tune_enable(False)
    yield force
    u1.set_pass_fusion(1)
    u1.tune_enable(True)


@pytest.mark.parametrize("dims,block", SHAPES)
def test_fp64_one_launch_sweep_parity(u1, orc, forced, dims, block):
    forced(dims, block, "f64")
    g, og, lat, ref = make_pair(u1, orc, dims, 0.9, 1.3, True, seed=59)
    say(f"fp64 one-launch sweep {dims} {block}")
    m, om = u1.metro(1, 3, 0.5), orc.metro(1, 3, 0.5)
    for s, (a, b) in enumerate(PASSES):
        assert lat.update(a, b, m, 59, s, count_accepts=True) == orc.update(og, ref, a, b, om, 59, s, count_accepts=True)
        assert np.array_equal(bits(lat.to_host()), bits(ref)), s
        p = lat.update_plaquette(a, b, m, 59, 8 + s)
        orc.update(og, ref, a, b, om, 59, 8 + s)
        assert np.array_equal(bits(lat.to_host()), bits(ref)), s
        assert np.max(np.abs(p - orc.plaquette(og, ref))) <= 1e-13


@pytest.mark.parametrize("dims,block", SHAPES)
def test_fp32_one_launch_sweep_matches_phases(u1, forced, dims, block):
    forced(dims, block, "f32")
    g = u1.geom(dims, 1.0, 1.2)
    out = {}
    for mode in (0, 1):  # pass fusion off: a launch per phase
        u1.set_pass_fusion(mode)
        lat = u1.Lattice.cold(g, u1.F32)
        lat.hotstart(29)
        acc = [lat.update(a, b, u1.BENCH_METRO, 29, s, count_accepts=True) for s, (a, b) in enumerate(PASSES)]
        p = [lat.update_plaquette(a, b, u1.BENCH_METRO, 29, 8 + s) for s, (a, b) in enumerate(PASSES)]
        out[mode] = (lat.to_host(), acc, np.array(p))
    say(f"fp32 one-launch sweep {dims} {block}: accepts {out[1][1]}")
    assert np.array_equal(out[0][0], out[1][0])
    assert out[0][1] == out[1][1]
    assert np.max(np.abs(out[0][2] - out[1][2])) <= 1e-12


@pytest.mark.parametrize("dims,block,ml", MASKED)
def test_fp64_one_launch_masked_sweep_parity(u1, orc, forced, dims, block, ml):
    forced(dims, block, "f64")
    g, og, lat, ref = make_pair(u1, orc, dims, 0.9, 1.3, True, seed=61)
    say(f"fp64 one-launch masked sweep {dims} {block} mask {ml}")
    m, om = u1.metro(1, 3, 0.5), orc.metro(1, 3, 0.5)
    for s, (a, b) in enumerate(PASSES):
        assert lat.update(a, b, m, 61, s, mask_ml=ml, count_accepts=True) == \
            orc.update(og, ref, a, b, om, 61, s, mask_ml=ml, count_accepts=True)
        assert np.array_equal(bits(lat.to_host()), bits(ref)), s


@pytest.mark.parametrize("dims,block,ml", MASKED + [((24, 24, 24, 8), 512, 2), ((24, 24, 24, 8), 1024, 2)])
def test_fp32_one_launch_masked_sweep_matches_phases(u1, forced, dims, block, ml):
    forced(dims, block, "f32")
    g = u1.geom(dims, 1.0, 1.2)
    out = {}
    for mode in (0, 1):
        u1.set_pass_fusion(mode)
        lat = u1.Lattice.cold(g, u1.F32)
        lat.hotstart(29)
        acc = [lat.update(a, b, u1.BENCH_METRO, 29, s, mask_ml=ml, count_accepts=True) for s, (a, b) in enumerate(PASSES)]
        out[mode] = (lat.to_host(), acc)
    say(f"fp32 one-launch masked sweep {dims} {block} mask {ml}: accepts {out[1][1]}")
    assert np.array_equal(out[0][0], out[1][0])
    assert out[0][1] == out[1][1]
