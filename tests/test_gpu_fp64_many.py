"""The FP64 kernels with a lane per target (k_accel64, k_field64), which take over
from k_rows64 and k_accel64sym for many targets: the bits of the oracle where a
chunk holds an extreme, subnormal or infinite coordinate (the general root and
quotient) beside chunks of ordinary ones, for wavefronts on, off and partly on the
cathode, and for the roles of the two-time-step update.

k_rows64 takes up to 2048 wavefronts of 64 targets by a chunk of 256 sources (half as
many without an image series), k_accel64sym 256 pairs of chunks or more of an
unbanded planar or tip simulation with image charges.  So 4100 particles without a series
(2210 of 2048), 5800 with one (2093, 253 pairs) and 6200 in the two-time-step mode
(2425) have a lane per target, and so have 22 000 and 44 000 points over 700
particles (2064)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NM = 1e-9
Q0, M0 = 1.602176634e-19, 9.1093837015e-31
TIP = (1000.0, 1000 * NM, 250 * NM, 500 * NM)
GEOMS = [("bare", 0), ("images", 0), ("images", 3), ("tip", 0)]


def _geom(dd, O, kind, nic):
    if kind == "tip":
        dd.set_tip(*TIP)
        return O.geom_tip(*TIP)
    dd.set_planar(2000.0, 1000 * NM, kind == "images", nic)
    return O.geom_planar(1000 * NM, 2000.0, kind == "images", nic)


def _cloud(n, kind, seed):
    rng = np.random.default_rng(seed)
    pos = np.stack([rng.uniform(-150, 150, n), rng.uniform(-150, 150, n),
                    rng.uniform(510 if kind == "tip" else 0.0, 990, n)], 1) * NM
    return pos, np.where(rng.uniform(size=n) < 0.2, Q0, -Q0), np.full(n, M0)


# (particle, coordinate, value): out of the ordinary range in the second chunk
ODD = [None, (300, 0, 3e-40), (300, 2, 1e-200), (300, 1, 1e40), (300, 0, np.inf)]


@pytest.mark.parametrize("odd", ODD)
@pytest.mark.parametrize("kind,nic", GEOMS)
def test_accelerations(oracle_mod, kind, nic, odd):
    from rumdeed_amd.diode import Diode

    n = 5800 if nic else 4100
    pos, q, m = _cloud(n, kind, 3)
    pos[900] = pos[20]  # coincident particles in different chunks
    if kind != "tip":
        pos[40, 2] = 0.0  # on the cathode: its n = 0 image is at its own place
    if odd:
        pos[odd[0], odd[1]] = odd[2]
    t = np.unique(np.concatenate([[0, 20, 40, 255, 256, 300, 511, 512, 900, n - 1],
                                  np.arange(7, n, 61)])).astype(np.int32)
    print(f"accel {kind} nic={nic} n={n} odd={odd}", flush=True)
    dd = Diode(n + 16)
    g = _geom(dd, oracle_mod, kind, nic)
    dd.put_particles(pos, q, m)
    a = dd.calculate_acceleration_particles("fp64")
    dd.set_partial_budget(24 * 5 * n)  # in bands of five chunks
    b = dd.calculate_acceleration_particles("fp64")
    dd.close()
    with np.errstate(all="ignore"):
        ref = oracle_mod.accel_subset(g, pos, q, m, t)
    assert np.array_equal(a[t], ref, equal_nan=True)
    assert np.array_equal(b, a, equal_nan=True)


@pytest.mark.parametrize("odd", ODD)
@pytest.mark.parametrize("kind,nic", GEOMS)
def test_field_points(oracle_mod, kind, nic, odd):
    from rumdeed_amd.diode import Diode

    n, m = 700, 44000 if nic else 22000
    pos, q, ms = _cloud(n, kind, 5)
    if odd:
        pos[odd[0], odd[1]] = odd[2]
    pts = _cloud(m, kind, 6)[0]
    if kind != "tip":
        pos[40, 2] = 0.0
        pts[64:128, 2] = 0.0   # a wavefront on the cathode
        pts[128:160, 2] = 0.0  # a wavefront partly on it
        pts[m - 64:, 2] = 0.0  # the last ones, a workgroup partly filled
        pts[m - 1, 2] = -0.0
    pts[70] = pos[40]          # points at particles' places
    pts[200] = pos[600]
    t = np.unique(np.concatenate([np.arange(60, 260), np.arange(m - 80, m), np.arange(0, m, 97)]))
    print(f"field {kind} nic={nic} m={m} odd={odd}", flush=True)
    dd = Diode(n + 16)
    g = _geom(dd, oracle_mod, kind, nic)
    dd.put_particles(pos, q, ms)
    f = dd.calc_field_at_batch(pts, "fp64")
    dd.close()
    with np.errstate(all="ignore"):
        ref = oracle_mod.field(g, pos, q, pts[t])
    assert np.array_equal(f[t], ref, equal_nan=True)


def test_two_time_step_roles(oracle_mod):
    from rumdeed_amd.diode import Diode

    n = 6200
    pos = _cloud(n, "images", 9)[0]
    sp = np.where(np.random.default_rng(n).random(n) < 0.5, 1, 2).astype(np.int32)
    dd = Diode(n + 8)
    so = oracle_mod.Sim(n + 8)
    so.set_geometry(_geom(dd, oracle_mod, "images", 2))
    for t in (dd, so):
        t.set_time_step(0.25e-15)
        t.set_two_time_step(2)
    dd.add_particles(pos, species=sp, step=1, emit=1)
    so.add(pos, species=sp, step=1, emit=1)
    for k in (1, 2):
        dd.update_position(k, "fp64")
        so.step(k, phases=2)
        sg, st = dd.get_state(), so.state()
        for f in ("pos", "vel", "acc"):
            assert np.array_equal(sg[f], st[f]), (k, f)
    dd.close()
