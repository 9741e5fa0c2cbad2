"""Jumps of more chains than the device holds workgroups for: workgroups that
wait for each other are started only where all of a launch's are resident, so no
wait passes a bound far above a jump's own time (2 ms against 0.4), however long
the simulations ahead of one take, and a step's jumps never run twice.  Records
and state are those of a launch per jump.

40 diodes of about 1000 chains need more than 64 chains in each of 512
workgroups; 24 of them fit with about 50, also with a dear image series."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NM = 1e-9
N, SIDE = 3400, 200.0


def _run(sims, nic, prec, one):
    from rumdeed_amd.diode import Pool

    rng = np.random.default_rng(5)
    z = NM + 999 * NM * rng.uniform(0, 1, N) ** 2
    pos = np.column_stack([rng.uniform(-SIDE / 2, SIDE / 2, N) * NM,
                           rng.uniform(-SIDE / 2, SIDE / 2, N) * NM, z])
    dd = Pool(sims * 6144, sims + 1)
    dd.set_solo_jumps(one)
    dd.set_jump_wait(2_000_000)
    slots = [dd.open(6144) for _ in range(sims)]
    for k, s in enumerate(slots):
        dd.select(s)
        dd.set_planar(8000.0, 1000 * NM, True, nic)
        dd.set_time_step(0.25e-15)
        dd.set_seed(3 + k)
        dd.set_emitter(10, 0, -SIDE / 2 * NM, -SIDE / 2 * NM, SIDE * NM, SIDE * NM,
                       wf=np.array([[4.7]]))
        dd.add_particles(pos)
    recs = dd.step(prec)
    out = [recs[s].as_dict() for s in slots]
    dd.select(slots[-1])
    st = dd.get_state()
    repeats = dd.jump_repeats()
    print(sims, nic, prec, "chains", sum(r["n_round"] for r in out), "repeats", repeats, flush=True)
    dd.close()
    return out, st["pos"], repeats


@pytest.mark.parametrize("sims,nic,prec", [(40, 0, "mixed"), (40, 10, "mixed"), (24, 10, "mixed"),
                                           (40, 2, "fp64")])
def test_waiting_workgroups_are_resident(sims, nic, prec):
    out, pos, repeats = _run(sims, nic, prec, True)
    assert sum(r["n_round"] for r in out) > 900 * sims
    assert repeats == 0
    apart, pos_apart, _ = _run(sims, nic, prec, False)
    assert out == apart
    assert np.array_equal(pos, pos_apart)
