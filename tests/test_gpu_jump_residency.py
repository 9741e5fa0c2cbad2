"""Jumps of more chains than the device holds workgroups for.

40 diodes of about 1000 chains need more than 64 chains in each of 256 (FP64) or 512
workgroups, 24 of them fit the mixed form with about 50; five of 3000 chains and
12 000 electrons with ten image terms took 138 workgroups each, of which the second
simulation's first ones then waited for the whole first simulation, past the
bound.  The launches are laid out so that no simulation waits longer than about
20 ms for its last workgroup's place: with a bound of 60 ms no wait gives up and no
step runs its jumps twice.  Uneven pools take more workgroups than places (small
simulations follow large ones).  Records and state are those of a launch per
jump."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NM = 1e-9


def _run(sizes, nic, prec, one):
    """One step of a pool of diodes of (electrons, side in nm)."""
    from rumdeed_amd.diode import Pool

    dd = Pool(sum(n + 2048 for n, _ in sizes) + 1024, len(sizes) + 1)
    dd.set_solo_jumps(one)
    dd.set_jump_wait(60_000_000)
    slots = [dd.open(n + 2048) for n, _ in sizes]
    for k, (s, (n, side)) in enumerate(zip(slots, sizes)):
        rng = np.random.default_rng(5 + k)
        z = NM + 999 * NM * rng.uniform(0, 1, n) ** 2
        dd.select(s)
        dd.set_planar(8000.0, 1000 * NM, True, nic)
        dd.set_time_step(0.25e-15)
        dd.set_seed(3 + k)
        dd.set_emitter(10, 0, -side / 2 * NM, -side / 2 * NM, side * NM, side * NM,
                       wf=np.array([[4.7]]))
        if n:
            dd.add_particles(np.column_stack([rng.uniform(-side / 2, side / 2, n) * NM,
                                              rng.uniform(-side / 2, side / 2, n) * NM, z]))
    recs = dd.step(prec)
    out = [recs[s].as_dict() for s in slots]
    states = []
    for s in (slots[0], slots[len(slots) // 2], slots[-1]):
        dd.select(s)
        states.append(dd.get_state()["pos"])
    repeats = dd.jump_repeats()
    print(len(sizes), nic, prec, "chains", sum(r["n_round"] for r in out), "repeats", repeats,
          flush=True)
    dd.close()
    return out, states, repeats


LIKE, LARGE = [(3400, 200.0)], [(12000, 370.0)]
UNEVEN = [(n, side) for n, side in ((9000, 170.0), (6000, 170.0), (3000, 150.0), (2000, 140.0),
                                    (1000, 130.0), (300, 120.0), (60, 100.0), (5, 80.0))
          for _ in range(8)] + [(0, 40.0)] * 8


@pytest.mark.parametrize("sizes,nic,prec", [(LARGE * 5, 10, "fp64"), (LIKE * 40, 1, "fp64"),
                                            (LIKE * 40, 0, "mixed"), (LIKE * 24, 10, "mixed"),
                                            (UNEVEN, 0, "fp64"), (UNEVEN, 0, "mixed"),
                                            (UNEVEN, 2, "mixed")])
def test_no_step_repeats_its_jumps(sizes, nic, prec):
    out, states, repeats = _run(sizes, nic, prec, True)
    assert sum(r["n_round"] for r in out) > 14000
    assert repeats == 0
    apart, states_apart, _ = _run(sizes, nic, prec, False)
    assert out == apart
    for a, b in zip(states, states_apart):
        assert np.array_equal(a, b)
