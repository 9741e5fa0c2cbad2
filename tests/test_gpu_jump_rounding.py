"""The squared height of a source enters the jumps' cathode distances unrounded.

As in test_gpu_field_rounding.py, two neighbouring FP32 heights whose squares
FP32 would round up and down by nearly half a step (6e-8), here just above 256 nm,
over an emitter beneath them (rho^2 at most a sixth of z^2).  The chains' fields show
in df_avg, the mean escape probability D: log D = -b w^(3/2) v / F is -3.7 at 8 GV/m
and 4.7 eV and falls 2.2 times as fast as 1/F there (v = 0.42 at l = 0.52), so a
relative error b of the source's part of the field, a share s of it, changes D by
8 b s.  A rounded square gives the two heights errors of +-8e-8, 1.6e-7 apart; the other
roundings (rms 1.4e-7 a term) average over 5000 chains to 2e-9 each, so the two
agree to 2e-8."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NM = 1e-9
Q0, M0 = 1.602176634e-19, 9.1093837015e-31
E0, GAP, SIDE, CHARGES = 8.0e9, 1000 * NM, 150 * NM, 256.0
SLOPE = 8.0  # d ln D / d ln F


def _heights():
    z = np.float32(256.0) + np.arange(1, 4000, dtype=np.float32) * np.float32(2.0 ** -15)
    step = (z.astype(np.float64) ** 2 - (z * z).astype(np.float64)) / 2.0 ** -7
    return float(z[np.argmax(step)]), float(z[np.argmin(step)]), step.max() - step.min()


def _df(prec, pool, z):
    from rumdeed_amd.diode import Diode, Pool

    if pool:
        dd = Pool(16384, 2)
        dd.open(8192)
    else:
        dd = Diode(8192)
    dd.set_planar(E0 * GAP, GAP, True, 0)
    dd.set_time_step(2.0e-15)
    dd.set_seed(5)
    dd.set_emitter(10, 0, -SIDE / 2, -SIDE / 2, SIDE, SIDE, wf=np.array([[4.7]]))
    dd.put_particles(np.array([[0.0, 0.0, z * NM]]), [-CHARGES * Q0], [M0])
    r = dd.do_emission(1, prec)
    dd.close()
    return r.df_avg, r.n_round


@pytest.mark.parametrize("pool", [False, True])
def test_squared_height(pool):
    zp, zm, apart = _heights()
    assert apart > 0.95
    share = 2 * CHARGES * Q0 / (4 * np.pi * 8.8541878128e-12 * (256 * NM) ** 2) / E0
    err = []
    for z in (zp, zm):
        d64, chains = _df("fp64", False, z)
        dm, cm = _df("mixed", pool, z)
        assert chains == cm > 4000
        err.append((dm / d64 - 1.0) / (SLOPE * share))
    print(zp, zm, "chains", chains, "share", share, err, flush=True)
    assert abs(err[0] - err[1]) < 2e-8
