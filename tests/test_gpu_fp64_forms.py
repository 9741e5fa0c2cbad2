"""The FP64 pair terms' fast root/quotient sequences and paired cathode form
against the oracle, bit for bit, where their rules could go wrong: a chunk
that holds an extreme, subnormal or infinite coordinate takes the general
sequences (the chunks beside it the fast ones), coincident particles, points
at a particle's place, wavefronts on, off and partly on the cathode, and the
edges of the 256-particle chunks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NM = 1e-9
Q0, M0 = 1.602176634e-19, 9.1093837015e-31
TIP = (1000.0, 1000 * NM, 250 * NM, 500 * NM)


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
    q = np.where(rng.uniform(size=n) < 0.2, Q0, -Q0)
    return pos, q, np.full(n, M0)


# (particle, coordinate, value): out of the ordinary range in the first chunk
ODD = [None, (7, 0, 3e-40), (7, 2, 1e-200), (7, 1, 1e40), (7, 0, np.inf)]


@pytest.mark.parametrize("odd", ODD)
@pytest.mark.parametrize("kind,nic", [("bare", 0), ("images", 0), ("images", 3), ("tip", 0)])
def test_extreme_coordinates(oracle_mod, kind, nic, odd):
    from rumdeed_amd.diode import Diode

    n = 700
    pos, q, m = _cloud(n, kind, 3)
    pos[300] = pos[20]  # coincident particles in different chunks
    if kind != "tip":
        pos[40, 2] = 0.0  # on the cathode: its n = 0 image is at its own place
    if odd:
        pos[odd[0], odd[1]] = odd[2]
    dd = Diode(n + 16)
    g = _geom(dd, oracle_mod, kind, nic)
    dd.put_particles(pos, q, m)
    print(f"accel {kind} nic={nic} odd={odd}", flush=True)
    a = dd.calculate_acceleration_particles("fp64")
    with np.errstate(all="ignore"):
        assert np.array_equal(a, oracle_mod.accel(g, pos, q, m), equal_nan=True)
    pts = _cloud(330, kind, 4)[0]
    if kind != "tip":
        pts[64:128, 2] = 0.0   # a wavefront on the cathode
        pts[128:160, 2] = 0.0  # a wavefront partly on it
    pts[70] = pos[40]          # points at particles' places
    pts[200] = pos[300]
    f = dd.calc_field_at_batch(pts, "fp64")
    with np.errstate(all="ignore"):
        assert np.array_equal(f, oracle_mod.field(g, pos, q, pts), equal_nan=True)
    dd.close()


@pytest.mark.parametrize("n", [1, 255, 256, 257, 513])
@pytest.mark.parametrize("m", [1, 63, 64, 65, 257])
def test_cathode_points_at_chunk_edges(oracle_mod, n, m):
    from rumdeed_amd.diode import Diode

    pos, q, ms = _cloud(n, "images", 5 + n)
    pts = _cloud(m, "images", 6 + m)[0]
    pts[:, 2] = 0.0
    pts[m // 2, 2] = -0.0
    dd = Diode(n + 16)
    for nic in (0, 1, 2):
        g = _geom(dd, oracle_mod, "images", nic)
        dd.put_particles(pos, q, ms)
        f = dd.calc_field_at_batch(pts, "fp64")
        assert np.array_equal(f, oracle_mod.field(g, pos, q, pts)), nic
    dd.close()
