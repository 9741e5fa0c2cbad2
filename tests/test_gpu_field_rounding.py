"""The squared height of a source enters the cathode field's distance unrounded.

Two heights a few FP32 steps apart, z+ and z-, are chosen so that rounding z^2 to
FP32 would raise one square and lower the other by nearly half a step (6e-8 of
z^2 just above 64 nm).  Beneath the electron z^2 is most of r^2, so with a rounded
square the mean relative errors of the field, 3/2 of that each with opposite
signs, would differ by more than 1e-7.  Every other rounding depends on the point as
well: over 8192 points the mean of errors of about 1.4e-7 has a standard deviation
of 1.6e-9, so the two means agree to 2e-8."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NM = 1e-9
Q0, M0 = 1.602176634e-19, 9.1093837015e-31


def _heights():
    z = np.float32(64.0) + np.arange(1, 4000, dtype=np.float32) * np.float32(2.0 ** -17)
    exact = z.astype(np.float64) ** 2
    step = (exact - (z * z).astype(np.float64)) / 2.0 ** -11  # FP32 step at 4096 .. 8192
    return float(z[np.argmax(step)]), float(z[np.argmin(step)]), step.max() - step.min()


@pytest.mark.parametrize("nic", [0, 2])
def test_squared_height(nic):
    from rumdeed_amd.diode import Diode

    zp, zm, apart = _heights()
    assert apart > 0.95
    rng = np.random.default_rng(8)
    rho, phi = rng.uniform(3.0, 20.0, 8192), rng.uniform(0, 2 * np.pi, 8192)
    pts = np.column_stack([rho * np.cos(phi), rho * np.sin(phi), 0 * rho]) * NM
    mean = []
    for z in (zp, zm):
        dd = Diode(16)
        dd.set_planar(2000.0, 1000 * NM, True, nic)
        dd.put_particles(np.array([[0.0, 0.0, z * NM]]), [-Q0], [M0])
        vacuum = -2000.0 / (1000 * NM)
        f64 = dd.calc_field_at_batch(pts, "fp64")[:, 2] - vacuum
        fm = dd.calc_field_at_batch(pts, "mixed")[:, 2] - vacuum
        dd.close()
        mean.append(np.mean((fm - f64) / f64))
    print(nic, zp, zm, mean, flush=True)
    assert abs(mean[0] - mean[1]) < 2e-8
