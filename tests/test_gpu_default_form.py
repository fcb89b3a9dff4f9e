"""The form a context starts with (a sweep direction fused with the RK update,
by the box's shape and size) against the separate form, bit for bit: sizes on
both sides of each limit, runs that end inside a group of enqueued steps (an
odd and an even number of idle ones) and go on, and an error stop."""
import numpy as np
import pytest

from hormone_amd import driver as D
from hormone_amd import problems as P
from hormone_amd.grid import cartesian_grid
from hormone_amd.native import Hydro, HgError, STOP_END

pytestmark = pytest.mark.gpu

CASES = [((130, 1, 1), True, 3), ((1, 67, 1), True, 2), ((1, 1, 67), False, 3),
         ((181, 181, 1), True, 3), ((182, 181, 1), True, 2), ((190, 1, 190), False, 3),
         ((1, 183, 183), True, 3), ((51, 50, 51), True, 3), ((51, 51, 52), False, 2),
         ((64, 33, 64), True, 1)]


def flow(n, mag, rk):
    prm = P.Params(n=n, mag_on=mag, rktype=rk, bc=(0,) * 12, courant=0.3, t_end=1e30,
                   dt_out=1e30, is_test=False)
    g = cartesian_grid(n, prm.lo, prm.hi)
    r = np.random.default_rng(5)

    def noise(a):
        return a * r.uniform(-1.0, 1.0, g.shape)
    st = P.State(d=1.0 + noise(0.2), p=1.0 + noise(0.2), v=[noise(0.3) for _ in range(3)],
                 b=[noise(0.3) * mag for _ in range(3)], phi=np.zeros(g.shape))
    return prm, g, st


def engine(prm, g, st, separate):
    eng = Hydro(**D.desc_fields(prm, g))
    if separate:
        eng.set_fused(0)
    D.load_initial_state(eng, prm, g, st)
    return eng


def fields(eng, prm, g):
    f = D.SNAP_FIELDS_MAG if prm.mag_on else D.SNAP_FIELDS
    return D.fetch(eng, g, f + tuple(D.F_U + q for q in range(eng.ufnmax())))


def same(a, b):
    for f in b:
        assert np.array_equal(a[f].view(np.uint64), b[f].view(np.uint64)), f


@pytest.mark.parametrize("n,mag,rk", CASES)
def test_gpu_default_form_equals_separate(hiplib, n, mag, rk):
    prm, g, st = flow(n, mag, rk)
    # when the run ends, after 5 and after 6 steps of the first group of 16
    ref = engine(prm, g, st, True)
    ends = [ref.run_loop(0.0, 0, 1e30, 1e30, 1e30, 2, 2, k, 1 << 40, 1 << 40, 0.5)[0]
            for k in (5, 6)]
    for end in ends:
        out = []
        for separate in (True, False):
            print(f"case default form n={n} mag={mag} rk={rk} separate={separate}", flush=True)
            eng = engine(prm, g, st, separate)
            t, tn, to, why = eng.run_loop(0.0, 0, 1e30, 1e30, end, 0, 1, 1 << 40, 1, 1 << 40, 0.5)
            assert why == STOP_END
            first = fields(eng, prm, g)
            # and on from there, in the run loop and call by call
            t, tn, to, why = eng.run_loop(t, tn, 1e30, 1e30, 1e30, 2, 2, 1 << 40, 1 << 40, 2, 0.5)
            dt, ch = eng.timestep(t, 1e30, 1e30, 2, 2)
            eng.hydro_step(dt, ch)
            out.append((t, tn, dt, ch, first, fields(eng, prm, g)))
        assert out[0][:4] == out[1][:4]
        same(out[1][4], out[0][4])
        same(out[1][5], out[0][5])


def test_gpu_default_form_stops_at_the_same_error(hiplib):
    prm, g, st = flow((182, 181, 1), True, 3)
    prm.courant = 3.0  # unstable: ends in a negative internal energy
    errs = []
    for separate in (True, False):
        print(f"case default form error separate={separate}", flush=True)
        eng = engine(prm, g, st, separate)
        with pytest.raises(HgError) as e:
            eng.run_loop(0.0, 0, 1e30, 1e30, 1e30, 2, 2, 1 << 40, 1 << 40, 400, 0.5)
        errs.append((e.value.code, e.value.cell, e.value.direction, e.value.tn, e.value.time))
    assert errs[0] == errs[1]
