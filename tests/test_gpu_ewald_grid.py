"""The gridded reciprocal sum (the path of large systems) against the direct
64-bit sum of the oracle, through mgpu_ewald: sizes just past the rule that
chooses it and larger, an ionic crystal (whose Bragg peaks meet the grid's
aliases) and a skewed cell, sites outside the box, sites on grid points, and
all sites crowded into a few bricks of the grid (more than a brick's bucket
holds).

Tolerances.  FP64: the oracle advances its phases by recurrence (lmax eps, about
25 x 1.1e-16) and adds the sites one after another (sqrt(N_s) eps, 160 x 1.1e-16,
each of its 2e4 terms), a few 1e-14 of the sums' terms, and the forces of neutral
molecules, of the crystal and of the cluster, and the energy beside the self
energy, are remainders of terms up to 100 times larger: 1e-11 and 5e-11.  Against
the sum in long double the grid is within 5e-15 in the forces.  Mixed: the FP32
weights and grid, 6e-8 a term, with the same remainders."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


def _system(name):
    from moldy_amd import system
    if name == "water":
        return system.water_box(3600, seed=11)
    if name == "skewed":
        s = system.water_box(8000, seed=12)
        L = s.h[0, 0]
        s.h = np.array([[L, 0.18 * L, -0.11 * L], [0.0, L, 0.14 * L], [0.0, 0.0, L]])
        return s
    if name == "salt":
        return system.salt_water(nwater=7500, nmg=137, ncl=274, seed=13)
    return system.silica(ncell=10, seed=14, cutoff=10.0)


def _past_rule(prec):
    """Just past the size rule of each precision."""
    from moldy_amd import engine as E, system
    return system.water_box(3600 if prec == E.FP64 else 5000, seed=11)


def _check(s, xyz, prec, tol_f, tol_e):
    from moldy_amd import engine as E
    from oracle.oracle import Oracle
    ref = Oracle(s).ewald(xyz)
    e = E.ForceEngine(s, precision=prec)
    f0 = np.random.default_rng(3).standard_normal((3, s.nsites))
    got = e.ewald(s.h, xyz, fxyz=f0.copy())
    again = e.ewald(s.h, xyz, fxyz=f0.copy())
    assert np.array_equal(got["force"], again["force"]) and got["pe"] == again["pe"]
    assert np.array_equal(got["stress"], again["stress"])
    assert got["info"].nhkl == ref["info"].nhkl
    scale = np.linalg.norm(ref["force"])
    err_f = np.linalg.norm(got["force"] - f0 - ref["force"]) / scale
    self_e = got["info"].self_energy
    err_e = abs(got["pe"] - ref["pe"]) / abs(ref["pe"] + self_e)
    err_s = rel_err(np.triu(got["stress"]), np.triu(ref["stress"]))
    print(f"{s.nsites} sites, {ref['info'].nhkl} k: force {err_f:.1e} energy {err_e:.1e} stress {err_s:.1e}", flush=True)
    assert err_f < tol_f and err_e < tol_e and err_s < tol_e
    e.close()


@pytest.mark.parametrize("name", ["water", "skewed", "salt", "silica"])
def test_fp64_vs_direct(name):
    from moldy_amd import engine as E
    from oracle.oracle import Oracle
    s = _system(name)
    _check(s, Oracle(s).make_sites(), E.FP64, 1e-11, 5e-11)


@pytest.mark.parametrize("name", ["skewed", "salt", "silica"])
def test_mixed_vs_direct(name):
    from moldy_amd import engine as E
    from oracle.oracle import Oracle
    s = _system(name)
    _check(s, Oracle(s).make_sites(), E.MIXED, 1e-5 if name == "silica" else 2e-6, 1e-6)


@pytest.mark.parametrize("case", ["outside", "on_points", "crowded"])
def test_placement(case):
    from moldy_amd import engine as E
    from oracle.oracle import Oracle
    s = _system("water")
    L = s.h[0, 0]
    xyz = Oracle(s).make_sites()
    if case == "outside":       # other periodic images, up to two boxes away
        xyz = xyz + L * np.random.default_rng(5).integers(-2, 3, xyz.shape)
    elif case == "on_points":   # multiples of L/16, the box's faces among them
        xyz = np.round(xyz * 16 / L) * L / 16
    else:                       # a cluster about a corner, across the periodic faces
        xyz = 0.02 * xyz + np.array([[0.5 * L], [-0.5 * L], [0.49 * L]])
    # the cluster's molecules are shrunk 50 times, and S(k) of neutral molecules
    # with them: a remainder 50 times smaller (forces), its square in the energy
    tol = (5e-10, 1e-7) if case == "crowded" else (1e-11, 5e-11)
    _check(s, np.ascontiguousarray(xyz), E.FP64, *tol)


def test_noalloc_takes_the_same_path():
    import test_zz_no_alloc as T
    T._compare(_system("water"), 6)


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("prec", [0, 1])
def test_coordinate_not_finite(bad, prec):
    """One site without a place makes every sum NaN, as in the direct sum (its
    phase enters every S(k)); the engine's next call is not touched by it."""
    from moldy_amd import engine as E
    from oracle.oracle import Oracle
    import test_zz_no_alloc as T
    s = _past_rule(prec)
    xyz = Oracle(s).make_sites()
    e = E.ForceEngine(s, precision=prec)
    zero = np.zeros((3, s.nsites))
    calls = ["mgpu_ewald"] + (["mgpu_ewald_noalloc"] if prec == E.FP64 else [])
    good = {}
    for name in calls:
        rc, f, pe, st, _ = T._call(e, name, s, xyz, zero)
        assert rc == 0 and np.all(np.isfinite(f)) and np.isfinite(pe)
        good[name] = (f, pe, st)
    for axis in range(3):
        x = xyz.copy()
        x[axis, 17 + axis] = bad
        for name in calls:
            rc, f, pe, st, _ = T._call(e, name, s, x, zero)
            assert rc == 0
            assert np.all(np.isnan(f)) and np.isnan(pe) and np.all(np.isnan(st[[0, 4, 8]])), (name, axis)
    for name in calls:
        rc, f, pe, st, _ = T._call(e, name, s, xyz, zero)
        assert np.array_equal(f, good[name][0]) and pe == good[name][1] and np.array_equal(st, good[name][2])
    e.close()
