"""All Metropolis-Hastings jumps of a step in one launch (k_mh_jumps64,
k_mh_jumps32) at the edges of their tiles.

The sums' order depends on the particle count and the kind of context alone,
so one launch and a launch per jump (rd_set_solo_jumps) give the same bits in
every form; FP64 equals the oracle.  Mixed against FP64: a field carries the
FP32 error of its space-charge part, here below 1e-8 of the field (a few
percent of it, each term good to about 1e-7), so an accept test (slope
d ln J / d ln F about 20) differs with probability 2e-7, 2e-3 over a case's
largest count of tests: the chains take the same sites, bit for bit.

Particle counts: the FP64 chunk (256), the particles the mixed forms hold in
LDS (1536, 2560) and the lone forms' switch (4096), each with its neighbours,
and few or none.  Emitter sides: about 1, 64 and 500 chains."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NM = 1e-9
INTS = ("n", "emitted", "n_round", "absorbed", "dropped", "start_rounds")
DBLS = ("n_sup", "ramo_current", "mh_std", "a_rate", "df_avg")
STATE = ("pos", "vel", "acc", "species", "section", "id")


def _particles(n, seed=11):
    rng = np.random.default_rng(seed + n)
    return np.column_stack([rng.uniform(-300, 300, n), rng.uniform(-300, 300, n),
                            rng.uniform(30, 180, n)]) * NM


def _setup(t, kind, side, n, oracle=None):
    """The same simulation on a Diode, a Pool's slot or the oracle."""
    ic, nic = {"none": (False, 0), "one": (True, 0), "series": (True, 2)}.get(kind, (True, 0))
    if kind == "tip":
        if oracle:
            t.set_geometry(oracle.geom_tip(1000.0, 1000 * NM, 250 * NM, 500 * NM, True), 1500 * NM)
        else:
            t.set_tip(1000.0, 1000 * NM, 250 * NM, 500 * NM, True, box_top=1500 * NM)
    elif oracle:
        t.set_geometry(oracle.geom_planar(200 * NM, 1600.0, ic, nic))
    else:
        t.set_planar(1600.0, 200 * NM, ic, nic)
    t.set_time_step(0.5e-15)
    t.set_seed(29)
    if kind == "tip":
        t.set_emitter(3, 0, w_tip=4.5)
    else:
        t.set_emitter(9 if kind == "gtf" else 10, 0, -side / 2 * NM, -side / 2 * NM, side * NM,
                      side * NM, T=1000.0, wf=np.array([[4.7]]))
    if n:
        p = _particles(n)
        if kind == "tip":
            p[:, 2] += 560 * NM
        (t.add if oracle else t.add_particles)(p)


def _run(kind, side, n, prec, pool, one, steps=2):
    from rumdeed_amd.diode import Diode, Pool

    if pool:
        dd = Pool(2 * 16384, 3)
        dd.open(16384)
    else:
        dd = Diode(16384)
    dd.set_solo_jumps(one)
    _setup(dd, kind, side, n)
    recs = [dd.step(prec)[0] for _ in range(steps)] if pool else dd.run(steps, prec)
    if pool:
        dd.select(0)
    st = dd.get_state()
    dd.close()
    print(kind, side, n, prec, "chains", [r.n_round for r in recs], "electrons",
          [r.n for r in recs], flush=True)
    return recs, st


def _same(a, b):
    for ra, rb in zip(a[0], b[0]):
        for f in INTS + DBLS:
            assert getattr(ra, f) == getattr(rb, f), f
        assert list(ra.f_avg) == list(rb.f_avg)
    for f in STATE:
        assert np.array_equal(a[1][f], b[1][f]), f


CASES = ([("one", 3, n) for n in (0, 1, 255, 257)] +
         [("one", 34, n) for n in (256, 1535, 1536, 1537, 2559, 2560, 2561, 4095, 4096, 4097)] +
         [("one", 110, 300), ("one", 110, 5000), ("series", 34, 513), ("series", 110, 1600),
          ("none", 34, 257), ("none", 3, 4100), ("gtf", 34, 700), ("tip", 0, 65)])


@pytest.mark.parametrize("kind,side,n", CASES)
def test_one_launch_equals_a_launch_per_jump(kind, side, n):
    for pool in (False, True):
        _same(_run(kind, side, n, "mixed", pool, True),
              _run(kind, side, n, "mixed", pool, False))
    _same(_run(kind, side, n, "fp64", False, True),
          _run(kind, side, n, "fp64", True, False))


@pytest.mark.parametrize("kind,side,n", [c for c in CASES if c[2] <= 1600 and c[0] != "tip"])
def test_fp64_jumps_equal_the_oracle(oracle_mod, kind, side, n):
    recs, st = _run(kind, side, n, "fp64", False, True)
    so = oracle_mod.Sim(16384, nthreads=8)
    _setup(so, kind, side, n, oracle_mod)
    ro = [so.step(k) for k in (1, 2)]
    _same((recs, st), (ro, so.state()))


@pytest.mark.parametrize("pool", [False, True])
@pytest.mark.parametrize("kind,side,n", [c for c in CASES if c[0] not in ("tip", "gtf")])
def test_mixed_jumps_take_the_sites_of_fp64(kind, side, n, pool):
    rm, sm = _run(kind, side, n, "mixed", pool, True, steps=1)
    rd, sd = _run(kind, side, n, "fp64", False, True, steps=1)
    for f in INTS:
        assert getattr(rm[0], f) == getattr(rd[0], f), f
    assert rm[0].mh_std == rd[0].mh_std
    k = len(sd["id"]) - rd[0].emitted  # the new electrons are the last rows
    assert np.array_equal(sm["pos"][k:, :2], sd["pos"][k:, :2])
