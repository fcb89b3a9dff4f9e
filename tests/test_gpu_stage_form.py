"""States between the stages of an x-fused step that hold conserved fields only
(boxes of more than 2^19 cells) against the separate form, bit for
bit: shapes on both sides of the limit, two and three stages, boundary codes
that take scalars and vectors from one cell and from different ones, self-gravity,
and a region so thin that its wavefronts fall back to plain division."""
import numpy as np
import pytest

from hormone_amd import driver as D
from hormone_amd import problems as P
from hormone_amd.grid import cartesian_grid
from hormone_amd.native import HgError, Hydro

pytestmark = pytest.mark.gpu

PER, REF, OUT, MIXED = (0,) * 12, (1,) * 12, (3,) * 6 + (2,) * 6, (1,) * 6 + (3,) * 6
CASES = [((80, 81, 80), True, 3, PER, 1.0), ((81, 81, 81), True, 3, PER, 1.0),
         ((81, 81, 81), True, 2, REF, 1.0), ((82, 80, 81), False, 3, OUT, 1.0),
         ((97, 131, 75), False, 2, REF, 1.0), ((81, 81, 81), True, 3, MIXED, 1.0),
         ((730, 721, 1), True, 3, OUT, 1.0), ((600001, 1, 1), True, 3, REF, 1.0),
         ((600001, 1, 1), False, 2, OUT, 1.0), ((81, 1, 7001), True, 3, PER, 1.0),
         ((81, 81, 81), True, 3, REF, 1e-90), ((81, 81, 81), False, 3, PER, 1e-90),
         ((81, 81, 81), True, 3, REF, -1e-90), ((81, 81, 81), False, 2, PER, -1e-90)]


def flow(n, mag, rk, bc, thin):
    prm = P.Params(n=n, mag_on=mag, rktype=rk, bc=bc, courant=0.3, t_end=1e30, dt_out=1e30,
                   is_test=False)
    g = cartesian_grid(n, prm.lo, prm.hi)
    r = np.random.default_rng(11)

    def noise(a):
        return a * r.uniform(-1.0, 1.0, g.shape)
    # a part of the box (all of it: negative) with density, pressure and B^2
    # scaled alike (same speeds)
    w = np.full(g.shape, abs(thin) if thin < 0.0 else 1.0)
    w.reshape(-1)[: w.size // 5] = abs(thin)
    st = P.State(d=w * (1.0 + noise(0.2)), p=w * (1.0 + noise(0.2)),
                 v=[noise(0.3) for _ in range(3)],
                 b=[np.sqrt(w) * noise(0.3) * mag for _ in range(3)], phi=np.zeros(g.shape))
    prm.thin = thin
    return prm, g, st


def fields(eng, prm, g):
    f = D.SNAP_FIELDS_MAG if prm.mag_on else D.SNAP_FIELDS
    return D.fetch(eng, g, f + (D.F_EINT,) + tuple(D.F_U + q for q in range(eng.ufnmax())))


def same(a, b):
    for f in b:
        assert np.array_equal(a[f].view(np.uint64), b[f].view(np.uint64)), f


def steps(eng, prm, g, st):
    D.load_initial_state(eng, prm, g, st)
    try:
        t, tn, to, why = eng.run_loop(0.0, 0, 1e30, 1e30, 1e30, 2, 2, 1 << 40, 1 << 40, 3, 0.5)
    except HgError as e:  # negative energy at the jump to the thin part (MHD)
        assert 0.0 < prm.thin < 1.0
        return {0: np.array([e.code, e.direction, *e.cell], dtype=np.float64)}
    dt, ch = eng.timestep(t, 1e30, 1e30, 2, 2)
    eng.hydro_step(dt, ch)
    return fields(eng, prm, g)


@pytest.mark.parametrize("n,mag,rk,bc,thin", CASES)
def test_gpu_x_fused_stage_form_equals_separate(hiplib, n, mag, rk, bc, thin):
    prm, g, st = flow(n, mag, rk, bc, thin)
    out = []
    for fused in (0, 2):
        print(f"case stage form n={n} mag={mag} rk={rk} bc={bc} thin={thin} fused={fused}",
              flush=True)
        eng = Hydro(**D.desc_fields(prm, g))
        eng.set_fused(fused)
        out.append(steps(eng, prm, g, st))
        eng.close()
    same(out[1], out[0])


@pytest.mark.parametrize("mag", [False, True], ids=["hydro", "mhd"])
def test_gpu_x_fused_stage_form_with_gravity(hiplib, mag):
    out = []
    for fused in (0, 2):
        print(f"case stage form gravity mag={mag} fused={fused}", flush=True)
        prm, g, st = P.make_problem("polytrope3d", n=82, steps=4, mag_on=mag)
        eng = Hydro(**D.desc_fields(prm, g))
        eng.set_fused(fused)
        D.load_initial_state(eng, prm, g, st)
        D.run(eng, prm, g, device_loop=True)
        out.append(fields(eng, prm, g))
        eng.close()
    same(out[1], out[0])
