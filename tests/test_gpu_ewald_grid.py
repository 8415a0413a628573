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


def _long_double_forces(s, xyz, pick):
    """The direct sum's forces on the sites pick, in long double throughout."""
    ld = np.longdouble
    assert np.array_equal(s.h, np.eye(3) * s.h[0, 0])
    L, al, kc = ld(s.h[0, 0]), ld(s.control.alpha), s.control.k_cutoff
    pi = ld("3.14159265358979323846264338327950288")
    b = 2 * pi / L
    m = int(kc / float(b))
    q = s.site_charges().astype(ld)
    fr = xyz.astype(ld) / L

    def powers(d, w):
        """w cos, w sin of 2 pi l f for l = 0 .. m"""
        ph = 2 * pi * ((np.arange(m + 1).astype(ld)[:, None] * fr[d][None]) % 1)
        return np.cos(ph) * w, np.sin(ph) * w
    one = np.ones_like(q)
    (cx, sx), (cy, sy), (cz, sz) = powers(0, one), powers(1, one), powers(2, q)
    F = np.zeros((3, len(pick)), ld)
    for h in range(m + 1):
        for k in range(-m if h else 0, m + 1):
            n2 = (kc / float(b)) ** 2 - h * h - k * k
            if n2 <= 0:
                continue
            # l and -l from the four real sums
            sk = np.sign(k) if k else 1
            c = cx[h] * cy[abs(k)] - sx[h] * sy[abs(k)] * sk
            t = sx[h] * cy[abs(k)] + cx[h] * sy[abs(k)] * sk
            nl = int(np.ceil(np.sqrt(n2)))
            cc, ss, cs, sc = cz[:nl] @ c, sz[:nl] @ t, sz[:nl] @ c, cz[:nl] @ t
            for l in range(-nl + 1 if (h or k) else 1, nl):
                a, g = abs(l), (1 if l >= 0 else -1)
                C, S = cc[a] - g * ss[a], sc[a] + g * cs[a]
                K = np.array([h * b, k * b, l * b])
                k2 = (K * K).sum()
                co = 8 * pi / L ** 3 * np.exp(-k2 / (4 * al * al)) / k2
                sin = t[pick] * cz[a, pick] + g * c[pick] * sz[a, pick]   # times q
                cos = c[pick] * cz[a, pick] - g * t[pick] * sz[a, pick]
                F += K[:, None] * (co * (C * sin - S * cos))[None]
    return F


@pytest.mark.parametrize("prec,nwater", [(0, 2800), (1, 4200)])
def test_forces_no_further_off_than_the_direct_sum(prec, nwater):
    """Ions in water, where the direct sum is closest: against the sum in long
    double it is 0.9e-15 (FP64) and 3.5e-7 (mixed) off at 4,054 sites and 1.7e-15 and
    5.4e-7 at 32,438.  The window's own part is 5e-16 and 1.4e-7, the rounding of
    weights, grid and transforms 1e-15 and 1e-7."""
    from moldy_amd import engine as E, system
    from oracle.oracle import Oracle
    s = system.salt_water(nwater=nwater, nmg=nwater // 55, ncl=2 * (nwater // 55), seed=13)
    xyz = Oracle(s).make_sites()
    pick = np.random.default_rng(2).choice(s.nsites, 100, replace=False)
    pick[:30] = np.arange(s.nsites - 30, s.nsites)     # ions
    e = E.ForceEngine(s, precision=prec)
    f = e.ewald(s.h, xyz)["force"][:, pick]
    e.close()
    if prec == E.FP64:
        ref = _long_double_forces(s, xyz, pick)
        err, tol = float(np.linalg.norm(f - ref) / np.linalg.norm(ref)), 1.5e-15
    else:
        err, tol = rel_err(f, Oracle(s).ewald(xyz)["force"][:, pick]), 2.4e-7
    print(f"{s.nsites} sites, precision {prec}: {err:.2e}", flush=True)
    assert err < tol


def test_molecular_forces_no_further_off_than_the_direct_sum():
    """The errors of a molecule's sites do not cancel on the grid as the direct
    sum's do (an error of S(k) is a smooth field): its molecular forces were
    1.086e-6 off at 32,438 sites, mixed against FP64."""
    from moldy_amd import engine as E, system
    s = system.salt_water(nwater=8000, nmg=146, ncl=292, seed=7)
    f = []
    for prec in (E.FP64, E.MIXED):
        e = E.ForceEngine(s, precision=prec)
        f.append(e.eval_forces())
        e.close()
    err = {k: rel_err(f[1][k], f[0][k]) for k in ("force", "torque", "site_force")}
    print({k: f"{v:.3e}" for k, v in err.items()}, flush=True)
    assert err["force"] < 1.086e-6 and err["torque"] < 1.109e-6 and err["site_force"] < 3.134e-7


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


def _took_grid(e):
    """Whether the last evaluation or ewald call with profiling on took the grid."""
    return e.profile_get("ewald_grid_spread")[1] > 0


def _route(s, prec):
    from moldy_amd import engine as E
    e = E.ForceEngine(s, precision=prec)
    e.profile(True)
    e.upload_state()
    e.eval_forces_device()
    grid = _took_grid(e)
    e.close()
    return grid


def _droplet(n, widen, alpha):
    """Liquid water in the middle of a box widen times wider."""
    from moldy_amd import system
    s = system.water_box(n, seed=3, alpha=alpha, cutoff=14.0)
    s.h = s.h * widen
    s.c_of_m = s.c_of_m / widen
    return s


def test_systems_of_these_tests_take_the_grid():
    from moldy_amd import engine as E, system
    for name in ("water", "skewed", "salt", "silica"):
        assert _route(_system(name), E.FP64), name
    for name in ("skewed", "salt", "silica"):
        assert _route(_system(name), E.MIXED), name
    for prec in (E.FP64, E.MIXED):
        assert _route(_past_rule(prec), prec)
    assert _route(system.salt_water(nwater=2800, nmg=50, ncl=100, seed=13), E.FP64)
    assert _route(system.salt_water(nwater=4200, nmg=76, ncl=152, seed=13), E.MIXED)
    # test_gpu_adjoint_grid.py's FP64 sides, and the replayed MD step's mixed one
    assert _route(system.water_box(3600, seed=31), E.FP64)
    assert _route(system.silica(ncell=7, seed=32, cutoff=10.0), E.FP64)
    assert _route(system.water_box(5000, seed=23), E.MIXED)


def test_full_bricks_of_a_droplet():
    """Bricks of 126 sites beside empty ones (the mean is 4): within the bucket
    that a dense liquid fills."""
    from moldy_amd import engine as E
    from oracle.oracle import Oracle
    s = _droplet(4000, 3.0, 0.15)
    assert _route(s, E.FP64)
    _check(s, Oracle(s).make_sites(), E.FP64, 1e-11, 5e-11)


@pytest.mark.parametrize("kind,prec,grid", [
    ("few sites, high cutoff", 1, False),     # 700 sites, a grid of 248^3
    ("few sites, high cutoff", 0, True),
    ("wide box", 1, False),                   # 4,000 sites in nine times their volume
    ("coarse droplet", 1, False),
    ("coarse liquid", 1, False),
    ("slab", 1, True),
])
def test_size_rule(kind, prec, grid):
    from moldy_amd import system
    if kind == "few sites, high cutoff":
        s = system.water_box(175, seed=3, alpha=3.0, cutoff=6.0)
    elif kind == "wide box":
        s = system.water_box(1000, seed=3)
        s.h = s.h * 3.0
    elif kind == "coarse droplet":
        s = _droplet(4000, 3.0, 0.15)
    elif kind == "coarse liquid":
        s = system.water_box(16000, seed=3, alpha=0.15, cutoff=18.0)
    else:
        s = system.water_box(8000, seed=3)
        s.h = s.h * np.array([1.0, 1.0, 3.0])
        s.c_of_m = s.c_of_m / np.array([1.0, 1.0, 3.0])
    assert _route(s, prec) == grid


@pytest.mark.parametrize("nwater,hmax", [(375, 36), (200, 40)])
def test_noalloc_takes_the_direct_sum_where_only_that_fits(nwater, hmax):
    """Few sites at a high cutoff: the grid needs 65 and 95 MiB, the direct sum 37
    and 48 of the 64."""
    from moldy_amd import engine as E, system
    from oracle.oracle import Oracle
    import test_zz_no_alloc as T
    s = system.water_box(nwater, seed=3, cutoff=6.0)
    s.control.k_cutoff = 2 * np.pi * (hmax + 0.5) / s.h[0, 0]
    s.control.alpha = s.control.k_cutoff / (2 * np.sqrt(-np.log(1e-6)))
    assert _route(s, E.FP64)
    xyz = Oracle(s).make_sites()
    f0 = np.random.default_rng(3).standard_normal((3, s.nsites))
    e = E.ForceEngine(s)
    rc, fa, pa, sa, ia = T._call(e, "mgpu_ewald_noalloc", s, xyz, f0)
    assert rc == 0, E.lib().mgpu_last_error(e.h_)
    rc, fb, pb, sb, ib = T._call(e, "mgpu_ewald", s, xyz, f0)
    assert rc == 0 and ia.hmax == ib.hmax == hmax
    e.close()
    # two sums of the same terms
    assert rel_err(fa - f0, fb - f0) < 1e-11
    assert abs(pa - pb) <= 5e-11 * (abs(pb) + ia.self_energy)
    assert rel_err(sa, sb) < 5e-11


def _flat(thin, order):
    """Water on a jittered 5 x 35 x 36 lattice, its thin side (24 grid points: three
    bricks, the fewest) along axis thin; 21 and 22 bricks (FP64), 18 and 19 (mixed)
    along the others."""
    from moldy_amd import system
    n = np.array(order)
    a = 2.9
    s = system.water_box(int(np.prod(n)), seed=9, cutoff=6.0)
    rng = np.random.default_rng(9)
    grid = np.stack(np.meshgrid(*[np.arange(k) for k in n], indexing="ij"), -1).reshape(-1, 3)
    pos = (grid + 0.5) / n - 0.5 + rng.normal(0, 0.1 / (a * n), grid.shape)
    s.c_of_m = pos - np.floor(pos + 0.5)
    s.h = np.diag(a * n)
    assert n[thin] == 5
    return s


@pytest.mark.parametrize("thin,order", [(0, (5, 35, 36)), (1, (36, 5, 35)), (2, (35, 36, 5))])
def test_flat_box(thin, order):
    from moldy_amd import engine as E
    from oracle.oracle import Oracle
    s = _flat(thin, order)
    xyz = Oracle(s).make_sites()
    for prec, tol in ((E.FP64, (1e-11, 5e-11)), (E.MIXED, (2e-6, 1e-6))):
        assert _route(s, prec)
        _check(s, xyz, prec, *tol)
