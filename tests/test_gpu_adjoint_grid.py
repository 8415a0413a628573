"""Charge derivatives through the gridded reciprocal sum (an FP64 engine past
the size rule) against the direct sum (the same engine in mixed precision,
whose adjoint is FP64 all the same): dE/dtheta, the cotangent product and the
directional derivative."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["water", "silica"])
def test_adjoint_grid_vs_direct(name):
    from moldy_amd import engine as E, system
    s = system.water_box(3600, seed=31) if name == "water" else system.silica(ncell=7, seed=32, cutoff=10.0)
    rng = np.random.default_rng(6)
    v = rng.standard_normal((3, s.nsites))
    th = E.get_theta(s)
    dth = rng.standard_normal(th.size) * np.abs(th)
    out = []
    for prec in (E.FP64, E.MIXED):
        e = E.ForceEngine(s, precision=prec)
        e.upload_state()
        out.append(e.adjoint(v=v, dtheta=dth))
        again = e.adjoint(v=v, dtheta=dth)
        assert all(np.array_equal(out[-1][k], again[k]) for k in ("dE", "vjp", "jvp"))
        e.close()
    a, b = out
    # sums of 1e4 sites and k vectors in two orders, few-fold cancellation
    for k in ("dE", "vjp", "jvp"):
        err = rel_err(a[k], b[k])
        print(name, k, f"{err:.1e}")
        assert err < 1e-11, k
    for k in ("dE", "vjp"):   # each charge's entry by itself
        q = slice(th.size - s.max_id, None)
        assert np.all(np.abs(a[k][q] - b[k][q]) <= 1e-10 * np.max(np.abs(b[k][q])))
