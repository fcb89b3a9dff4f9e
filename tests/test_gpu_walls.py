"""Walls and quiet gas in the FP64 sweeps: ghosts whose momentum or field is a
zero of the other sign (reflecting and outgoing walls), and velocities, fields
and psi that fall off to nothing ahead of a front, against the oracle bit for
bit; and that neither sends the sweeps through their plain form as well."""
import numpy as np
import pytest

from hormone_amd import driver as D
from hormone_amd import problems as P
from hormone_amd.grid import cartesian_grid
from hormone_amd.native import Hydro
from oracle.pyoracle import Oracle

pytestmark = pytest.mark.gpu

PER, REF, OUT = (0,) * 12, (1,) * 12, (2,) * 12
APART = (1, 2, 2, 1, 1, 1, 2, 1, 1, 2, 2, 2)


def flow(kind, n, mag, bc, limiter="modified_mc", seed=7):
    prm = P.Params(n=n, mag_on=mag, bc=bc, courant=0.3, t_end=1e30, dt_out=1e30, is_test=False)
    prm.flux_limiter = limiter
    g = cartesian_grid(n, prm.lo, prm.hi)
    r = np.random.default_rng(seed)
    sh = g.shape

    def noise(a):
        return a * r.uniform(-1.0, 1.0, sh)

    def zeros():
        return np.where(r.uniform(size=sh) < 0.3, -0.0, 0.0)
    d, p = 1.0 + noise(0.2), 1.0 + noise(0.2)
    v, b = [noise(0.3) for _ in range(3)], [noise(0.3) * mag for _ in range(3)]
    phi = noise(0.1) * mag
    if kind == "rest":          # nothing moves, and no field across any wall
        v, b = [np.zeros(sh) for _ in range(3)], [np.zeros(sh) for _ in range(3)]
    elif kind == "in":          # through every upper face, out of every lower one
        v = [-abs(x) for x in v]
    elif kind == "signed":      # zeros of both signs among the values
        v = [np.where(r.uniform(size=sh) < 0.5, zeros(), x) for x in v]
        b = [np.where(r.uniform(size=sh) < 0.5, zeros(), x) * mag for x in b]
        phi = np.where(r.uniform(size=sh) < 0.5, zeros(), phi) * mag
    elif kind == "front":       # falling off to 2^-400 from one corner to the other
        at = sum(np.linspace(0.0, 1.0, m).reshape([-1 if q == a else 1 for q in range(3)])
                 for a, m in enumerate(sh)) / 3.0
        v, b, phi = [x * np.exp2(-400.0 * at) for x in v], [x * np.exp2(-400.0 * at) for x in b], \
            phi * np.exp2(-400.0 * at)
    elif kind.startswith("tail"):  # exponents down to 2^-low, with gaps of 0
        low = float(kind[4:])

        def tail(x):
            x = x * np.exp2(-r.uniform(0.0, low, sh))
            return np.where(r.uniform(size=sh) < 0.2, 0.0, x)
        v, b, phi = [tail(x) for x in v], [tail(x) for x in b], tail(phi)
        if low < 500:
            d, p = np.ones(sh), np.ones(sh)
    return prm, g, P.State(d=d, p=p, v=v, b=b, phi=phi)


def steps(eng, prm, g, st):
    D.load_initial_state(eng, prm, g, st)
    dt, ch = eng.timestep(0.0, 1e30, 1e30, 2, 2)
    for _ in range(2):
        eng.hydro_step(dt, ch)
    return D.fetch(eng, g, D.SNAP_FIELDS_MAG if prm.mag_on else D.SNAP_FIELDS)


KINDS = ["rest", "in", "signed", "front", "tail300", "tail440", "tail700", "tail1070"]


@pytest.mark.parametrize("bc", [REF, OUT, APART, PER], ids=["reflecting", "outgoing", "apart",
                                                           "periodic"])
@pytest.mark.parametrize("mag,limiter,n", [(True, "modified_mc", (37, 9, 1)),
                                           (True, "minmod", (9, 5, 33)),
                                           (False, "modified_mc", (9, 37, 5)),
                                           (False, "flat", (70, 1, 1)),
                                           (True, "modified_mc", (1, 21, 8)),
                                           (True, "flat", (67, 4, 3))])
def test_gpu_walls_match_oracle(hiplib, mag, limiter, n, bc):
    for kind in KINDS:
        prm, g, st = flow(kind, n, mag, bc, limiter)
        want = steps(Oracle(**D.desc_fields(prm, g)), prm, g, st)
        for fused in (0, 1, 2):
            if fused and n[{1: 2 if n[2] > 1 else 1, 2: 0}[fused]] == 1:
                continue
            print(f"case walls {kind} mag={mag} {limiter} n={n} bc={bc} fused={fused}", flush=True)
            eng = Hydro(**D.desc_fields(prm, g))
            eng.set_fused(fused)
            got = steps(eng, prm, g, st)
            for f, x in want.items():
                assert np.array_equal(got[f].view(np.uint64), x.view(np.uint64)), (kind, f)
            eng.close()


def test_gpu_walls_with_conserved_stages_match_separate(hiplib):
    """The same in a box that keeps only conserved fields between its stages."""
    for kind, bc in (("rest", REF), ("signed", OUT), ("tail440", REF), ("tail1070", PER)):
        for mag in (False, True):
            prm, g, st = flow(kind, (81, 81, 81), mag, bc)
            out = []
            for fused in (0, 2):
                print(f"case walls 81^3 {kind} mag={mag} bc={bc} fused={fused}", flush=True)
                eng = Hydro(**D.desc_fields(prm, g))
                eng.set_fused(fused)
                out.append(steps(eng, prm, g, st))
                eng.close()
            for f, x in out[0].items():
                assert np.array_equal(out[1][f].view(np.uint64), x.view(np.uint64)), (kind, f)


def test_gpu_gravity_keeps_signed_zeros(hiplib):
    """With self-gravity a momentum of -0 may show the sign of a zero flux."""
    prm, g, st = P.make_problem("polytrope3d", n=20, steps=2)
    prm.bc = REF
    r = np.random.default_rng(3)
    st.v = [np.where(r.uniform(size=g.shape) < 0.5, -0.0, 0.0) for _ in range(3)]
    st.extra["grvphi_padded"] = np.zeros_like(st.extra["grvphi_padded"])
    st.d, st.p = np.ones(g.shape), np.ones(g.shape)
    out = []
    for cls in (Oracle, Hydro):
        print(f"case gravity signed zeros {cls.__name__}", flush=True)
        eng = cls(**D.desc_fields(prm, g))
        D.load_initial_state(eng, prm, g, st)
        D.run(eng, prm, g)
        out.append(D.fetch(eng, g, D.SNAP_FIELDS))
    for f, x in out[0].items():
        assert np.array_equal(out[1][f].view(np.uint64), x.view(np.uint64)), f


def sweep_ms(kind, mag, bc):
    prm, g, st = flow(kind, (56, 56, 56), mag, bc)
    eng = Hydro(**D.desc_fields(prm, g))
    D.load_initial_state(eng, prm, g, st)
    eng.timestep(0.0, 1e30, 1e30, 2, 2)
    eng.time_sweep(50)
    best = min(eng.time_sweep(100) for _ in range(7))
    eng.close()
    return best


@pytest.mark.parametrize("mag", [False, True], ids=["hydro", "mhd"])
@pytest.mark.parametrize("kind,bc", [("rest", REF), ("in", OUT), ("front", PER)])
def test_gpu_walls_cost_no_second_form(hiplib, kind, bc, mag):
    """Every wavefront of a box this size holds ghosts.  Running the plain form
    after the fast one takes at least half as long again; the boundary codes
    themselves take a few operations in the ghost lanes."""
    print(f"case walls time {kind} mag={mag}", flush=True)
    assert sweep_ms(kind, mag, bc) < 1.25 * sweep_ms("plain", mag, PER)
