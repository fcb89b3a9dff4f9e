"""Fields come back from the device as they went there, for the fields that
are staged in one piece and those that are staged in chunks (3 MB and more),
with rows and chunks that do not divide evenly; ghost cells of the caller's
array stay as they are."""
import numpy as np
import pytest

from hormone_amd import driver as D
from hormone_amd import problems as P
from hormone_amd.grid import cartesian_grid
from hormone_amd.native import Hydro

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (64, 64, 95), (64, 64, 96), (97, 131, 75), (1, 1, 400003), (400003, 1, 1),
          (3, 100003, 2), (130, 127, 129)]


@pytest.mark.parametrize("n", SHAPES)
def test_gpu_download_returns_what_was_uploaded(hiplib, n):
    print(f"case download n={n}", flush=True)
    prm = P.Params(n=n, mag_on=False, bc=(1,) * 12, t_end=1.0, dt_out=1.0, is_test=False,
                   gravswitch=3, grktype=2)
    g = cartesian_grid(n, prm.lo, prm.hi)
    eng = Hydro(**D.desc_fields(prm, g))
    r = np.random.default_rng(3)
    up = {f: g.pad(r.uniform(1.0, 2.0, g.shape)) for f in (D.F_D, D.F_E)}
    up.update({f: g.pad(r.uniform(-0.5, 0.5, g.shape)) for f in (D.F_V1, D.F_GRVPSI)})
    up.update({f: g.pad(np.zeros(g.shape)) for f in (D.F_V2, D.F_V3)})
    up[D.F_GRVPHI] = r.normal(size=g.padded_shape)
    for f, a in up.items():
        eng.upload(f, a)
    inner = tuple(slice(2, 2 + m) for m in g.shape)

    def get(f):
        a = np.full(g.padded_shape, -7.0)
        eng.download(f, a)
        b = a[inner].copy()
        a[inner] = -7.0
        assert (a == -7.0).all(), "ghost cells written"
        return b

    for f, a in up.items():
        assert np.array_equal(get(f), a[inner]), f
    assert np.array_equal(get(D.F_P), (prm.gamma - 1.0) * get(D.F_EINT))
    eng.close()
