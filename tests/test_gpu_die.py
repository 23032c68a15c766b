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


@pytest.fixture
def forced(u1, tmp_path):
    def force(dims, block, suffix):
        vol = "x".join(map(str, dims))
        rows = [f"{vol}\tSweep{a}+{b}_{suffix}\tthreads=halfvolume\t{block}\t1\t1\t0\t1\t1\t0\t# forced" for a, b in PASSES]
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
