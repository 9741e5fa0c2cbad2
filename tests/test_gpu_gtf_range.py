"""The thermal-field current at the small end of the double range: its quotients take
the general IEEE sequence where a numerator is so small that the residual of the
short one would be subnormal, so the supply equals the oracle's bit for bit.

Fields, temperatures (1 to 160 K) and work functions whose current density lies
between 1e-312 and 1e-270 A/m^2; an emitter and a time step of that size of no
diode keep the supply itself (current x area x time / charge) a normal number."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GAP, SIDE, DT = 1.0e-6, 1.0e-3, 1.0


def test_supply_of_tiny_currents(oracle_mod):
    from rumdeed_amd.diode import Diode

    rng = np.random.default_rng(1)
    dd = Diode(1024)
    bad, seen = [], 0
    while seen < 300:
        T, F, w = 10 ** rng.uniform(0, 2.2), -10 ** rng.uniform(6.5, 8.2), rng.uniform(2.0, 5.5)
        J = oracle_mod.gtf(F, T, w)
        if not 1e-312 < J < 1e-270:
            continue
        seen += 1
        so = oracle_mod.Sim(1024, nthreads=4)
        so.set_geometry(oracle_mod.geom_planar(GAP, -F * GAP, False, 0))
        dd.set_planar(-F * GAP, GAP, False, 0)
        for t in (dd, so):
            t.set_time_step(DT)
            t.set_seed(1)
            t.set_emitter(9, 0, -SIDE / 2, -SIDE / 2, SIDE, SIDE, T=T, wf=np.array([[w]]))
        a, b = dd.do_emission(1, "fp64").n_sup, so.step(1, phases=1).n_sup
        assert 0.0 < b < 1e-230
        if a != b:
            bad.append((F, T, w, a, b))
    dd.close()
    print(len(bad), "of", seen, "differ", bad[:3], flush=True)
    assert not bad
