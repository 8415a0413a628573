"""Shells of 129 to 256 z-columns (small subcells): the balanced kernel's form
with four groups of columns, at both ends of its range and with the largest
potential table (16 ids; FP64 then needs more than 64 KiB of LDS a block),
against the oracle and, mixed, against the walk; and grouped replica launches of it."""
import numpy as np
import pytest

from conftest import rel_err
import systems_small as S

pytestmark = pytest.mark.gpu


def _system(subcell, ids, nwater=400, seed=12):
    from moldy_amd import system
    s = system.salt_water(nwater=nwater, nmg=8, ncl=16, seed=seed, cutoff=7.0, alpha=0.38)
    s.control.subcell = subcell
    if ids > s.max_id:      # ids without sites
        pp = system.empty_potpar(ids)
        pp[:s.max_id, :s.max_id] = s.potpar
        s.potpar = pp
        s.site_mass = np.concatenate([s.site_mass, np.zeros(ids - len(s.site_mass))])
        s.site_charge = np.concatenate([s.site_charge, np.zeros(ids - len(s.site_charge))])
    return s


def _columns(s):
    from oracle.oracle import Oracle
    o = Oracle(s)
    off = np.asarray(o.neighbour_offsets()).reshape(-1, 3)
    half = {(int(x), int(y)) for x, y, _ in off}
    return len(half | {(-x, -y) for x, y in half})


# (subcell, ids, columns at least, at most)
WIDE = [(1.0, 6, 129, 192), (0.8, 6, 193, 256), (0.8, 16, 214, 256)]


@pytest.mark.parametrize("mode", [2, 3])
@pytest.mark.parametrize("subcell,ids,lo,hi", WIDE)
def test_wide_shells(subcell, ids, lo, hi, mode):
    from moldy_amd import engine as E
    from oracle.oracle import Oracle
    s = _system(subcell, ids)
    assert lo <= _columns(s) <= hi
    o = Oracle(s)
    xyz = o.make_sites()
    ref = o.force_calc(xyz)
    for prec in (E.FP64, E.MIXED):
        e = E.ForceEngine(s, precision=prec)
        e.set_realspace_mode(1)
        walk = e.force_calc(s.h, xyz)
        assert not e.realspace_balanced()
        e.set_realspace_mode(mode)
        got = e.force_calc(s.h, xyz)
        assert e.realspace_balanced()
        r, tol = (ref, 1e-10) if prec == E.FP64 else (walk, 1e-6)
        assert rel_err(got["force"], r["force"]) < tol
        assert rel_err(np.triu(got["stress"]), np.triu(r["stress"])) < tol
        # FP32 energies of cancelling Coulomb terms: as the mixed tests have it
        assert abs(got["pe"] - r["pe"]) <= (tol if prec == E.FP64 else 1e-4) * abs(r["pe"])
        e.close()


@pytest.mark.parametrize("prec", [0, 1])
def test_wide_shells_grouped(prec):
    """Replicas of uneven size stepped by grouped launches, against each alone."""
    from moldy_amd import engine as E, system
    if prec == E.FP64:
        sys_ = [S.two_species_generic(1, seed=21, n=150), S.two_species_generic(1, seed=22, n=200)]
        for s in sys_:     # no charges: FP64 Ewald steps have no grouped launches
            s.site_charge[:] = 0.0
            s.control.alpha = -1.0
            s.control.subcell = 0.75
    else:
        sys_ = [_system(0.8, 16), _system(0.8, 16, nwater=420, seed=17)]
    dyn = system.Dynamics(step=1e-4, temp=0.0, const_temp=0)
    res = []
    for batch in (True, False):
        es = []
        for s in sys_:
            e = E.ForceEngine(s, precision=prec)
            e.set_realspace_mode(2)
            e.set_dynamics(dyn)
            e.upload_state()
            e.upload_momenta(*s.thermal_momenta(50.0, seed=5))
            es.append(e)
        if batch:
            b = E.Batch(es)
            b.steps(4, init_H_0=True, schedule=E.SCHED_GROUPED)
            b.close()
        else:
            for e in es:
                e.md_steps(4, init_H_0=True)
        assert all(e.realspace_balanced() for e in es)
        res.append([e.download_dynamics() for e in es])
        for e in es:
            e.close()
    assert all(128 < _columns(s) <= 256 for s in sys_)
    for a, b in zip(*res):
        assert np.all(np.isfinite(a["mom"]))
        assert all(np.array_equal(a[k], b[k]) for k in ("c_of_m", "quat", "mom", "amom"))
