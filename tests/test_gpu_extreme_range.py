"""The sweeps' checked fast divisions and square roots, and the plain form a
wavefront takes where an operand is out of their range: states of extreme
exponent and negative zeros, in all or in a few of the cells, against the
oracle bit for bit."""
import numpy as np
import pytest

from hormone_amd import driver as D
from hormone_amd import problems as P
from hormone_amd.grid import cartesian_grid
from hormone_amd.native import Hydro
from oracle.pyoracle import Oracle

pytestmark = pytest.mark.gpu


def state(kind, n, mag, seed=11):
    """A smooth periodic flow with noise, then what `kind` does to it."""
    prm = P.Params(n=n, mag_on=mag, bc=(0,) * 12, t_end=1e30, dt_out=1e30, is_test=False)
    g = cartesian_grid(n, prm.lo, prm.hi)
    r = np.random.default_rng(seed)
    sh = g.shape

    def noise(a):
        return a * r.uniform(-1.0, 1.0, sh)
    d, p = 1.0 + noise(0.3), 1.0 + noise(0.3)
    v, b = [noise(0.5) for _ in range(3)], [noise(0.5) * mag for _ in range(3)]
    few = r.uniform(size=sh) < 0.02
    if kind == "small_units":      # every value far below the fast range
        d, p, b = d * 2.0 ** -300, p * 2.0 ** -300, [x * 2.0 ** -150 for x in b]
    elif kind == "large_units":
        d, p, b = d * 2.0 ** 300, p * 2.0 ** 300, [x * 2.0 ** 150 for x in b]
    elif kind == "tiny_components":  # nonzero, but far below the rest
        v[2] = v[2] * 1e-250
        b[1] = b[1] * 1e-290
    elif kind == "few_tiny":
        v[1] = np.where(few, v[1] * 1e-200, v[1])
        b[2] = np.where(few, 1e-310, b[2]) * mag
    elif kind == "negative_zero":
        v[0] = np.full(sh, -0.0)
        b[0] = np.full(sh, -0.0 if mag else 0.0)
    elif kind == "few_negative_zero":
        v[2] = np.where(few, -0.0, 0.0)
    elif kind == "uniform":         # zero slopes, zero radicands and dividends
        d, p = np.ones(sh), np.ones(sh)
        v = [np.zeros(sh) for _ in range(3)]
        b = [np.ones(sh) * mag, np.zeros(sh), np.zeros(sh)]
    return prm, g, P.State(d=d, p=p, v=v, b=b, phi=np.zeros(sh))


KINDS = ["plain", "small_units", "large_units", "tiny_components", "few_tiny", "negative_zero",
         "few_negative_zero", "uniform"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("mag,limiter,n", [(True, "modified_mc", (37, 9, 1)),
                                           (True, "minmod", (9, 5, 33)),
                                           (False, "modified_mc", (9, 37, 5)),
                                           (False, "flat", (70, 1, 1)),
                                           (True, "flat", (1, 21, 8))])
def test_gpu_extreme_values_match_oracle(hiplib, kind, mag, limiter, n):
    prm, g, st = state(kind, n, mag)
    prm.flux_limiter = limiter
    outs = []
    for cls, fused in ((Oracle, 0), (Hydro, 0), (Hydro, 2)):
        if fused and n[0] == 1:
            continue
        print(f"case {kind} mag={mag} {limiter} n={n} {cls.__name__} fused={fused}", flush=True)
        eng = cls(**D.desc_fields(prm, g))
        if fused:
            eng.set_fused(fused)
        D.load_initial_state(eng, prm, g, st)
        dt, ch = eng.timestep(0.0, 1e30, 1e30, 2, 2)
        for _ in range(2):
            eng.hydro_step(dt, ch)
        outs.append(D.fetch(eng, g, D.SNAP_FIELDS_MAG if mag else D.SNAP_FIELDS))
    for got in outs[1:]:
        for f, want in outs[0].items():
            assert np.array_equal(got[f].view(np.uint64), want.view(np.uint64)), f
