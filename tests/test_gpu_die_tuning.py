"""The choice of one-launch sweeps, with and without the plaquette: each is tuned for
itself, and without tuning a measured sweep goes by its own entry or else by the plain
sweep's.  The lattice does not depend on it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DIMS = (6, 4, 4, 6)
HEAD = "tunecache\tlatticeu1_amd-1\tgpu_arch=gfx950\nvolume\tname\taux\n"


def sweeps(u1, path):
    u1.tune_save(str(path))
    vol = "x".join(map(str, DIMS)) + "\t"
    rows = [ln.split("\t") for ln in path.read_text().splitlines() if ln.startswith(vol) and "\tSweep2+1" in ln]
    return {r[1]: int(r[3]) for r in rows}


def test_measured_sweeps_have_their_own_choice(u1, tmp_path):
    out = []
    for tune in (True, False):
        u1.tune_enable(tune)
        try:
            lat = u1.Lattice.cold(u1.geom(DIMS, 1.0), u1.F64)
            lat.hotstart(11)
            p = lat.update_plaquette(2, 1, u1.BENCH_METRO, 11, 0)
            if tune:
                assert set(sweeps(u1, tmp_path / "a.csv")) == {"Sweep2+1Plaq_f64"}
                lat2 = u1.Lattice.cold(u1.geom(DIMS, 1.0), u1.F64)
                lat2.hotstart(11)
                lat2.update(2, 1, u1.BENCH_METRO, 11, 0)
                assert set(sweeps(u1, tmp_path / "b.csv")) == {"Sweep2+1Plaq_f64", "Sweep2+1_f64"}
                assert np.array_equal(lat.to_host(), lat2.to_host())
            out.append((lat.to_host(), p))
        finally:
            u1.tune_enable(True)
        # without tuning: a launch per phase for the measured sweep, whatever the plain entry says
        row = "x".join(map(str, DIMS)) + "\t%s\tthreads=halfvolume\t%d\t1\t1\t0\t1\t1\t0\t# forced\n"
        f = tmp_path / "c.csv"
        f.write_text(HEAD + row % ("Sweep2+1_f64", 128) + row % ("Sweep2+1Plaq_f64", 0))
        u1.tune_load(str(f))
    assert np.array_equal(out[0][0], out[1][0])
    assert np.max(np.abs(out[0][1] - out[1][1])) <= 1e-13
