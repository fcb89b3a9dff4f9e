"""The bytes hg_profile_read reports for a launch against bench.py's model, for
boxes on both sides of the size from which only conserved fields are kept
between the stages, and for boundary codes that rule that out."""
import pytest

import bench
from hormone_amd import driver as D
from hormone_amd import native
from hormone_amd import problems as P
from hormone_amd.grid import cartesian_grid
from hormone_amd.native import Hydro

pytestmark = pytest.mark.gpu

PER, APART = (0,) * 12, (1,) * 6 + (3,) * 6
CASES = [((80, 81, 80), True, 3, PER, "fp64", 2, False),
         ((81, 81, 81), True, 3, PER, "fp64", 2, True),
         ((81, 81, 81), True, 2, PER, "fp64", 2, True),
         ((81, 81, 81), False, 3, PER, "fp64", 2, True),
         ((81, 81, 81), False, 3, APART, "fp64", 2, False),
         ((81, 81, 81), True, 3, PER, "fp32mix", 2, False),
         ((81, 81, 81), True, 3, PER, "fp64", 1, False),
         ((81, 81, 81), True, 3, PER, "fp64", 0, False),
         ((730, 721, 1), True, 3, PER, "fp64", 2, True),
         ((600001, 1, 1), False, 2, PER, "fp64", 2, True)]


@pytest.mark.parametrize("n,mag,rk,bc,precision,fused,conserved", CASES)
def test_gpu_profile_bytes_match_the_model(hiplib, n, mag, rk, bc, precision, fused, conserved):
    print(f"case profile bytes n={n} mag={mag} rk={rk} {precision} fused={fused}", flush=True)
    prm = P.Params(n=n, mag_on=mag, rktype=rk, bc=bc, precision=precision, is_test=False)
    eng = Hydro(**D.desc_fields(prm, cartesian_grid(n, prm.lo, prm.hi)))
    eng.set_fused(fused)
    nv, nw, dim = eng.ufnmax(), 10 if mag else 6, sum(m > 1 for m in n)
    sweep, update = bench.kernel_bytes(fused, nv, nw, dim, mag, rk, conserved)
    cells = n[0] * n[1] * n[2]
    assert eng.profile_read(native.PROF_SWEEP)[2] == pytest.approx(sweep * cells, rel=1e-12)
    assert eng.profile_read(native.PROF_RK)[2] == pytest.approx(update * cells, rel=1e-12)
    eng.close()
