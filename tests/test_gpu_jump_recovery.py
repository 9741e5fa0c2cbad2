"""Jumps of a step repeated after a workgroup's wait gave up.

The waits of the one-launch jumps are bounded; a bound of zero
(rd_set_jump_wait) makes the first workgroup that arrives give up, one of a few
microseconds lets some jumps through, so that workgroups leave at different
jumps with counters, widths and result arrays half written.  Every kernel ends
by itself, the host repeats the jumps with a launch per jump, and records and
state are those of an undisturbed run, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NM = 1e-9
FIELDS = ("n", "emitted", "n_round", "absorbed", "dropped", "n_sup", "ramo_current", "mh_std",
          "a_rate", "df_avg")
STATE = ("pos", "vel", "acc", "species", "section", "id")
STEPS = 3


def _setup(dd, k):
    side = (140.0, 90.0, 120.0)[k]
    rng = np.random.default_rng(3 + k)
    n = (900, 300, 500)[k]
    dd.set_planar(1600.0, 200 * NM, True, 1 if k == 1 else 0)
    dd.set_time_step(0.5e-15)
    dd.set_seed(17 + k)
    # the third one, thermal-field, waits for nobody
    dd.set_emitter(9 if k == 2 else 10, 0, -side / 2 * NM, -side / 2 * NM, side * NM, side * NM,
                   T=1000.0, wf=np.array([[4.7]]))
    dd.add_particles(np.column_stack([rng.uniform(-side / 2, side / 2, n),
                                      rng.uniform(-side / 2, side / 2, n),
                                      rng.uniform(30, 180, n)]) * NM)


def _run(prec, pool, graphs, wait, one=True):
    from rumdeed_amd.diode import Diode, Pool

    if pool:
        dd = Pool(3 * 8192, 4)
        slots = []
        for k in range(3):
            slots.append(dd.open(8192))
            _setup(dd, k)
    else:
        dd = Diode(8192)
        _setup(dd, 0)
    dd.set_graphs(graphs)
    dd.set_jump_wait(wait)
    dd.set_solo_jumps(one)
    print(prec, "pool" if pool else "lone", "graphs" if graphs else "", "wait", wait, flush=True)
    if pool:
        recs = []
        for _ in range(STEPS):
            rr = dd.step(prec)
            recs += [rr[s] for s in slots]
    else:
        recs = dd.run(STEPS, prec)
    states = []
    for s in (slots if pool else [None]):
        if pool:
            dd.select(s)
        states.append(dd.get_state())
    repeats = dd.jump_repeats()
    dd.close()
    assert min(r.n_round for r in recs[:2 if pool else 1]) > 64  # several workgroups
    return [[getattr(r, f) for f in FIELDS] for r in recs], states, repeats


@pytest.mark.parametrize("graphs", [False, True])
@pytest.mark.parametrize("pool", [False, True])
@pytest.mark.parametrize("prec", ["mixed", "fp64"])
def test_repeated_jumps_equal_an_undisturbed_run(prec, pool, graphs):
    recs, states, repeats = _run(prec, pool, graphs, -1)
    assert repeats == 0
    for wait in (0, 2000, 5000):
        r, s, repeats = _run(prec, pool, graphs, wait)
        print("repeats", repeats, flush=True)
        assert repeats == STEPS or wait > 0
        assert r == recs
        for a, b in zip(states, s):
            for f in STATE:
                assert np.array_equal(a[f], b[f]), f


@pytest.mark.parametrize("pool", [False, True])
@pytest.mark.parametrize("prec", ["mixed", "fp64"])
def test_graphs_leave_a_launch_per_jump_alone(prec, pool):
    assert _run(prec, pool, True, -1, one=False)[0] == _run(prec, pool, False, -1)[0]


def test_arguments():
    import ctypes

    from rumdeed_amd import _lib as L

    lib = L.lib()
    v = ctypes.c_int64()
    assert lib.rd_set_jump_wait(None, 0) == 1
    assert lib.rd_jump_repeats(None, ctypes.byref(v)) == 1
