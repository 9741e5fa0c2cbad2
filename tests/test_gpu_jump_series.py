"""The jump kernel of the planar image series and of diodes without image charges
(jump_planar): its particle rounds (256, lone from 4096 particles 1024), passes of
eight, four, two and one chains, and pools that hold all its forms.

The terms are those of the kernel's FP64 twin to a few FP32 roundings, so the
chains take the same sites (test_gpu_jumps.py derives the probability of
another), and a simulation gives the same bits alone in a pool and beside
others."""
import numpy as np
import pytest

from test_gpu_jumps import INTS, NM, STATE, _particles, _run, _same

pytestmark = pytest.mark.gpu

# emitter sides: about 1, 6, 15, 64 and 500 chains
CASES = ([("series", s, n) for s, n in ((3, 1), (9, 63), (14, 65), (20, 255), (34, 257), (34, 4097),
                                        (110, 1023), (110, 4500))] +
         [("none", s, n) for s, n in ((9, 64), (14, 256), (34, 1025), (110, 4096))])


@pytest.mark.parametrize("kind,side,n", CASES)
def test_sites_and_launches(kind, side, n):
    rd, sd = _run(kind, side, n, "fp64", False, True, steps=1)
    k = len(sd["id"]) - rd[0].emitted  # the new electrons are the last rows
    for pool in (False, True):
        one = _run(kind, side, n, "mixed", pool, True, steps=1)
        _same(one, _run(kind, side, n, "mixed", pool, False, steps=1))
        for f in INTS:
            assert getattr(one[0][0], f) == getattr(rd[0], f), f
        assert np.array_equal(one[1]["pos"][k:, :2], sd["pos"][k:, :2])


def test_all_forms_of_a_pool():
    from rumdeed_amd.diode import Pool

    forms = [(True, 0, 60, 700), (True, 10, 60, 300), (False, 0, 60, 500), (True, 1, 110, 900),
             (None, 0, 0, 200)]  # the last one a tip

    def setup(dd, k):
        ic, nic, side, n = forms[k]
        p = _particles(n, 50 + k)
        if ic is None:
            dd.set_tip(1000.0, 1000 * NM, 250 * NM, 500 * NM, True, box_top=1500 * NM)
            p[:, 2] += 560 * NM
        else:
            dd.set_planar(1600.0, 200 * NM, ic, nic)
        dd.set_time_step(0.5e-15)
        dd.set_seed(70 + k)
        if ic is None:
            dd.set_emitter(3, 0, w_tip=4.5)
        else:
            dd.set_emitter(10, 0, -side / 2 * NM, -side / 2 * NM, side * NM, side * NM,
                           wf=np.array([[4.7]]))
        dd.add_particles(p)

    def run(which):
        dd = Pool(8192 * len(which), len(which) + 1)
        slots = [dd.open(8192) for _ in which]
        for s, k in zip(slots, which):
            dd.select(s)
            setup(dd, k)
        recs = [dd.step("mixed") for _ in range(2)]
        out = {}
        for s, k in zip(slots, which):
            dd.select(s)
            st = dd.get_state()
            out[k] = ([r[s].as_dict() for r in recs], [st[f] for f in STATE])
        dd.close()
        return out

    both = run(range(len(forms)))
    for k in range(len(forms)):
        alone = run([k])[k]
        print(forms[k], "chains", alone[0][0]["n_round"], flush=True)
        assert alone[0] == both[k][0], forms[k]
        for a, b in zip(alone[1], both[k][1]):
            assert np.array_equal(a, b), forms[k]
