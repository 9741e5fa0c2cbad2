"""The mixed pair kernels at the edges of their tiles and rules, against the
FP64 kernels (which equal the oracle bit for bit).

A sum of terms each good to a few FP32 roundings is within 1e-6 of the sum of
the terms' magnitudes S (the oracle's scale).  Gather form: 64 targets and
quarters (64) of 256-source chunks; pair-symmetric: blocks of 256 and 512, one
and two targets per lane, from 5120 particles with image partners n >= 1, from
12 288 without.  Charges of both forms' loops: electrons only, and uneven."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NM = 1e-9
Q0, M0 = 1.602176634e-19, 9.1093837015e-31
TOL = 1e-6


def _cloud(n, tip, even, seed=5):
    rng = np.random.default_rng(seed + n)
    pos = np.column_stack([rng.uniform(-150, 150, n), rng.uniform(-150, 150, n),
                           rng.uniform(550 if tip else 1, 950, n)]) * NM
    q = np.full(n, -Q0) if even else -Q0 * rng.choice([1.0, 2.0, 0.5], n)
    return pos, q, np.full(n, M0)


def _open(geom, n, oracle):
    from rumdeed_amd.diode import Diode

    dd = Diode(n + 8)
    if geom == "tip":
        dd.set_tip(1000.0, 1000 * NM, 250 * NM, 500 * NM, True)
        return dd, oracle.geom_tip(1000.0, 1000 * NM, 250 * NM, 500 * NM, True)
    ic, nic = {"none": (False, 0), "one": (True, 0), "series": (True, 1), "far": (True, 4)}[geom]
    dd.set_planar(2000.0, 1000 * NM, ic, nic)
    return dd, oracle.geom_planar(1000 * NM, 2000.0, ic, nic)


SMALL = [1, 2, 63, 64, 65, 255, 256, 257, 700]
CASES = ([(g, n) for g in ("none", "one", "series", "far", "tip") for n in SMALL] +
         [("series", n) for n in (5119, 5120, 5377, 49152, 49153)] +
         [("one", n) for n in (12287, 12288, 12545, 28671, 28672)] + [("none", 12288), ("far", 5130)])


@pytest.mark.parametrize("even", [True, False])
@pytest.mark.parametrize("geom,n", CASES)
def test_accelerations(oracle_mod, geom, n, even):
    pos, q, m = _cloud(n, geom == "tip", even)
    dd, g = _open(geom, n, oracle_mod)
    dd.put_particles(pos, q, m)
    a64 = dd.calculate_acceleration_particles("fp64")
    am = dd.calculate_acceleration_particles("mixed")
    dd.close()
    t = np.unique(np.linspace(0, n - 1, min(n, 300)).astype(int))
    s = oracle_mod.accel_scale(g, pos, q, m, t)
    assert (np.linalg.norm(am[t] - a64[t], axis=1) <= TOL * s).all()


@pytest.mark.parametrize("geom", ["none", "one", "series", "far", "tip"])
@pytest.mark.parametrize("m,n", [(1, 1), (1, 257), (63, 65), (64, 256), (65, 700), (300, 3000),
                                 (5000, 13000)])
@pytest.mark.parametrize("surface", [False, True])
def test_field_points(oracle_mod, geom, m, n, surface):
    pos, q, mass = _cloud(n, geom == "tip", m != 300)
    pts = _cloud(m + 1, geom == "tip", True, 99)[0][:m]
    if surface and geom != "tip":
        pts[:, 2] = 0.0
        if m == 65:
            pts[64, 2] = 4 * NM  # one wavefront on the cathode, one off it
    dd, g = _open(geom, n, oracle_mod)
    dd.put_particles(pos, q, mass)
    f64 = dd.calc_field_at_batch(pts, "fp64")
    fm = dd.calc_field_at_batch(pts, "mixed")
    dd.close()
    t = np.unique(np.linspace(0, m - 1, min(m, 300)).astype(int))
    s = oracle_mod.field_scale(g, pos, q, pts[t])
    assert (np.linalg.norm(fm[t] - f64[t], axis=1) <= TOL * s).all()
