"""MD steps on the gridded reciprocal sum: the barostat (the plan follows the
cell every step: the k set's box changes on the way, and with every strain free
the cell leaves the triangular form) against the oracle, and replicas past the
size rule under every schedule against each alone."""
import numpy as np
import pytest

from conftest import rel_err
from moldy_amd import system

pytestmark = pytest.mark.gpu

TOL = 1e-10     # two sums of the same terms over four steps: up to 1.3e-12 (the energy beside its self term)


def _engine(s, dyn, precision, T=350.0, seed=3):
    from moldy_amd import engine as E
    e = E.ForceEngine(s, precision=precision)
    e.set_dynamics(dyn)
    e.upload_state()
    e.upload_momenta(*s.thermal_momenta(T, seed=seed))
    return e


def _gridded(e):
    e.profile(True)
    e.upload_state()
    e.eval_forces_device()
    g = e.profile_get("ewald_grid_spread")[1] > 0
    e.profile(False)
    return g


@pytest.mark.parametrize("name,mode,mask,npt", [("pr", 1, 200, False), ("free", 1, 0, True), ("uniform", 2, 200, True)])
def test_barostat_vs_oracle(name, mode, mask, npt):
    from moldy_amd import units
    from oracle.oracle import Oracle
    s = system.water_box(3600, seed=11)
    # |h| reaches 16 at the start and 15 once the cell has shrunk by 2e-5
    s.control.k_cutoff = 2 * np.pi * 16.0003 / s.h[0, 0]
    dyn = system.Dynamics(step=0.0005, pmass=10.0, const_pressure=mode, pressure=2e4 / units.CONV_P,
                          strain_mask=mask, temp=350.0 if npt else 0.0, const_temp=int(npt), ttmass=50.0)
    nsteps = 4
    step, st = Oracle(s).md(dyn, *s.thermal_momenta(350.0, seed=3))
    rec = []
    for i in range(nsteps):
        rc, pe, stress, r = step(i == 0)
        assert rc == 0
        rec.append(r[:8])
    e = _engine(s, dyn, 0)
    assert _gridded(e)
    h0 = e.last_info()[1].hmax
    e.upload_state()
    e.upload_momenta(*s.thermal_momenta(350.0, seed=3))
    tr1, _, _ = e.md_steps(2, init_H_0=True)
    tr2, pe_g, st_g = e.md_steps(nsteps - 2)
    got = e.download_dynamics()
    h, hmom = e.download_cell()
    errs = dict(trace=rel_err(np.vstack([tr1, tr2]), rec), pe=rel_err(pe_g, pe), stress=rel_err(st_g, stress),
                h=rel_err(h, st["h"]), hmom=rel_err(hmom, st["hmom"]),
                **{k: rel_err(got[k], st[k]) for k in ("c_of_m", "quat", "mom", "amom")})
    print(name, {k: f"{v:.1e}" for k, v in errs.items()}, "h", h.tolist(), "hmax", h0, e.last_info()[1].hmax)
    assert all(v < TOL for v in errs.values()), errs
    assert h0 == 16 and e.last_info()[1].hmax == 15
    lower = h[[1, 2, 2], [0, 0, 1]]
    assert np.all(lower != 0.0) if mask == 0 else np.all(lower == 0.0)
    e.close()


@pytest.mark.parametrize("schedule", [0, 1, 2, 3])
def test_replicas_past_the_rule(schedule):
    from moldy_amd import engine as E
    dyn = system.Dynamics(step=0.0005, temp=0.0, const_temp=0)
    reps = [system.water_box(5000, seed=41), system.water_box(343, seed=42), system.water_box(5600, seed=43)]
    res = []
    for batch in (False, True):
        es = [_engine(s, dyn, E.MIXED, T=300.0, seed=k) for k, s in enumerate(reps)]
        assert [_gridded(e) for e in es] == [True, False, True]
        out = []
        b = E.Batch(es) if batch else None
        for n, init in ((3, True), (2, False)):
            if batch:
                tr = list(b.steps(n, init_H_0=init, schedule=schedule))
            else:
                tr = [e.md_steps(n, init_H_0=init, use_graph=False)[0] for e in es]
            out.append((tr, [e.download_dynamics() for e in es]))
        if b:
            b.close()
        for e in es:
            e.close()
        res.append(out)
    for (ta, da), (tb, db) in zip(*res):
        for r in range(len(reps)):
            assert np.all(np.isfinite(ta[r])) and np.array_equal(ta[r], tb[r]), r
            assert all(np.array_equal(da[r][k], db[r][k]) for k in ("c_of_m", "quat", "mom", "amom")), r
