"""The mixed pair-symmetric accelerations at the edges of their blocks (256 and
512 particles, one and two targets per lane) against the FP64 kernels, within 1e-6 of
the terms' magnitudes S as in test_gpu_mixed_forms.py; and the argument check of
rd_set_jump_pairing."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NM = 1e-9
Q0, M0 = 1.602176634e-19, 9.1093837015e-31


@pytest.mark.parametrize("even", [True, False])
@pytest.mark.parametrize("nic,n", [(1, 5377), (4, 5633), (1, 49665), (0, 12545), (0, 28673)])
def test_block_edges(oracle_mod, nic, n, even):
    from rumdeed_amd.diode import Diode

    rng = np.random.default_rng(n)
    pos = np.column_stack([rng.uniform(-150, 150, n), rng.uniform(-150, 150, n),
                           rng.uniform(1, 950, n)]) * NM
    q = np.full(n, -Q0) if even else -Q0 * rng.choice([1.0, 2.0, 0.5], n)
    m = np.full(n, M0)
    dd = Diode(n + 8)
    dd.set_planar(2000.0, 1000 * NM, True, nic)
    dd.put_particles(pos, q, m)
    a64 = dd.calculate_acceleration_particles("fp64")
    am = dd.calculate_acceleration_particles("mixed")
    dd.close()
    edges = [k + o for k in (64, 128, 256, 512, 1024, 5120, n // 512 * 512, n // 256 * 256)
             for o in (-1, 0, 1)]
    t = np.unique([0, n - 2, n - 1] + [k for k in edges if 0 <= k < n]).astype(np.int32)
    s = oracle_mod.accel_scale(oracle_mod.geom_planar(1000 * NM, 2000.0, True, nic), pos, q, m, t)
    assert (np.linalg.norm(am[t] - a64[t], axis=1) <= 1e-6 * s).all()


def test_pairing_threshold_is_checked():
    from rumdeed_amd._lib import RumdeedError
    from rumdeed_amd.diode import Diode

    dd = Diode(64)
    for v in (0, 1 << 40):
        dd.set_jump_pairing(v)
    with pytest.raises(RumdeedError, match="negative"):
        dd.set_jump_pairing(-1)
    dd.close()
