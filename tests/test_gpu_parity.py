"""GPU parity: the HIP engine against the CPU oracle on identical inputs.

Bit-exact: cell assignment, cell list order, site neighbour lists.
FP64 path: forces, energies and virial within 1e-10 relative (norm-wise).
"""
import numpy as np
import pytest

from conftest import rel_err
import systems_small as S

pytestmark = pytest.mark.gpu

TOL64 = 1e-10


@pytest.fixture(scope="module")
def eng_mod():
    from moldy_amd import engine
    return engine


def _oracle(s):
    from oracle.oracle import Oracle
    return Oracle(s)


CASES = {
    "water": lambda: S.water(),
    "water_strict": lambda: _strict(S.water()),
    "water_molpbc": lambda: _molpbc(S.water()),
    "salt": S.salt,
    "argon_strict": lambda: S.argon(True),
    "argon": lambda: S.argon(False),
    "silica": S.silica,
    "clay": lambda: S.example("clay")[0],
    "mgclh2o": lambda: _mgcl(),
    # skewed cells: the hexagonal quartz example (Buckingham + Ewald, h01 < 0)
    # and water in a cell with h01, h02 and h12 all nonzero
    "quartz": lambda: S.example_auto("quartz")[0],
    "sheared_water": lambda: S.sheared_water(),
    # the surface-dipole term (src/accel.c:542-558) with a large total dipole
    "water_dipole": lambda: _dipole(S.water()),
    "salt_dipole": lambda: _dipole(S.salt()),
}


def _dipole(s):
    """Surface dipole on; even waters turned to molecule 0's orientation and
    odd ones to molecule 1's, so the total dipole (and the term) is large."""
    s.control.surface_dipole = True
    s.quat[0::2] = s.quat[0]
    s.quat[1::2] = s.quat[1]
    return s


def _strict(s):
    s.control.strict_cutoff = True
    return s


def _molpbc(s):
    s.control.molpbc = True
    return s


def _mgcl():
    s, e = S.example("mgclh2o")
    # positions from a seeded lattice (the logged run used a random start)
    rng = np.random.Generator(np.random.Philox(3))
    n = s.nmols
    g = int(np.ceil(n ** (1 / 3)))
    grid = np.stack(np.meshgrid(*[np.arange(g)] * 3, indexing="ij"), -1).reshape(-1, 3)
    pick = rng.permutation(len(grid))[:n]
    s.c_of_m = (grid[pick] + 0.5) / g - 0.5
    from moldy_amd.system import random_quaternions
    s.quat = random_quaternions(rng, s.nmols_r)
    s.h = np.eye(3) * 18.76756976
    return s


@pytest.mark.parametrize("case", list(CASES))
def test_cells_bit_exact(eng_mod, case):
    s = CASES[case]()
    o = _oracle(s)
    xyz = o.make_sites()
    ref = o.fill_cells(xyz)
    e = eng_mod.ForceEngine(s)
    got = e.cells(s.h, xyz)
    assert got["dims"] == ref["dims"]
    assert np.array_equal(got["entry_cell"], ref["entry_cell"])
    assert np.array_equal(got["cell_start"], ref["cell_start"])
    assert np.array_equal(got["cell_entries"], ref["cell_entries"])
    e.close()


@pytest.mark.parametrize("case", list(CASES))
def test_pairlist_bit_exact(eng_mod, case):
    s = CASES[case]()
    o = _oracle(s)
    xyz = o.make_sites()
    ref = o.site_lists(xyz)
    e = eng_mod.ForceEngine(s)
    got = e.pairlist(s.h, xyz)
    assert np.array_equal(got["start"], ref["start"])
    assert np.array_equal(got["nab"], ref["nab"])
    assert np.array_equal(got["pbctrans"], ref["pbctrans"])
    assert np.array_equal(got["nfnab"], ref["nfnab"])
    e.close()


@pytest.mark.parametrize("case", list(CASES))
def test_force_calc_fp64(eng_mod, case):
    s = CASES[case]()
    o = _oracle(s)
    xyz = o.make_sites()
    ref = o.force_calc(xyz)
    assert ref["rc"] == 0
    e = eng_mod.ForceEngine(s)
    got = e.force_calc(s.h, xyz)
    assert rel_err(got["force"], ref["force"]) < TOL64
    assert abs(got["pe"] - ref["pe"]) <= TOL64 * max(abs(ref["pe"]), 1e-300)
    assert rel_err(np.triu(got["stress"]), np.triu(ref["stress"])) < TOL64
    assert got["info"].n_too_close == ref["info"].n_too_close
    assert got["info"].nx == ref["info"].nx and got["info"].n_nabors == ref["info"].n_nabors
    e.close()


# systems whose shell splits into z-columns of cells (the clay's shell does
# not, and falls back to the per-offset walk in either mode)
BALANCED_CASES = tuple(c for c in CASES if c != "clay")


@pytest.mark.parametrize("mode", [1, 2, 3, 4])
@pytest.mark.parametrize("case", list(CASES))
def test_force_calc_fp64_both_kernels(eng_mod, case, mode):
    """The per-offset walk (1), the load-balanced kernel, candidates placed
    in windows of 2048 (2) or of 64 (3), and the column-tiled
    kernel (4), each against the oracle: same pair set, forces, energy,
    virial and close-pair count."""
    s = CASES[case]()
    o = _oracle(s)
    xyz = o.make_sites()
    ref = o.force_calc(xyz)
    e = eng_mod.ForceEngine(s)
    e.set_realspace_mode(mode)
    got = e.force_calc(s.h, xyz)
    assert e.realspace_balanced() == (mode >= 2 and case in BALANCED_CASES)
    assert rel_err(got["force"], ref["force"]) < TOL64
    assert abs(got["pe"] - ref["pe"]) <= TOL64 * max(abs(ref["pe"]), 1e-300)
    assert rel_err(np.triu(got["stress"]), np.triu(ref["stress"])) < TOL64
    assert got["info"].n_too_close == ref["info"].n_too_close
    e.close()


@pytest.mark.parametrize("case", BALANCED_CASES)
def test_mixed_realspace_kernels_agree(eng_mod, case):
    """In FP32 the real-space kernels differ only in summation order."""
    s = CASES[case]()
    out = []
    for mode in (1, 2, 3, 4):
        e = eng_mod.ForceEngine(s, precision=1)
        e.set_realspace_mode(mode)
        e.upload_state()
        pe, dip, st = e.eval_forces_device()
        assert e.realspace_balanced() == (mode >= 2)
        out.append((pe.copy(), st.copy(), e.download()[3].copy()))
        e.close()
    pa, sa, fa = out[0]
    for pb, sb, fb in out[1:]:
        assert rel_err(fb, fa) < 1e-6
        assert rel_err(sb, sa) < 1e-6
        assert np.max(np.abs(pb - pa)) <= 1e-6 * np.max(np.abs(pa))


@pytest.mark.parametrize("case", [c for c in CASES if not c.startswith("argon")])
def test_ewald_fp64(eng_mod, case):
    s = CASES[case]()
    o = _oracle(s)
    xyz = o.make_sites()
    ref = o.ewald(xyz)
    e = eng_mod.ForceEngine(s)
    got = e.ewald(s.h, xyz)
    assert got["info"].nhkl == ref["info"].nhkl
    assert rel_err(got["force"], ref["force"]) < TOL64
    assert abs(got["pe"] - ref["pe"]) <= TOL64 * abs(ref["pe"])
    assert rel_err(np.triu(got["stress"]), np.triu(ref["stress"])) < TOL64
    e.close()


@pytest.mark.parametrize("case", list(CASES))
def test_eval_forces_fp64(eng_mod, case):
    s = CASES[case]()
    o = _oracle(s)
    ref = o.eval_forces()
    assert ref["rc"] == 0
    e = eng_mod.ForceEngine(s)
    got = e.eval_forces()
    assert np.allclose(got["site_xyz"], ref["site_xyz"], rtol=0, atol=1e-12)
    assert rel_err(got["site_force"], ref["site_force"]) < TOL64
    assert rel_err(got["force"], ref["force"]) < TOL64
    if s.nmols_r:
        assert rel_err(got["torque"], ref["torque"]) < TOL64
    for k in range(2):
        assert abs(got["pe"][k] - ref["pe"][k]) <= TOL64 * max(abs(ref["pe"][k]), 1e-300)
    assert rel_err(got["stress"], ref["stress"]) < TOL64
    assert rel_err(got["dip"], ref["dip"]) < TOL64 or np.linalg.norm(ref["dip"]) < 1e-9
    e.close()


@pytest.mark.parametrize("ptype", [0, 1, 2, 3, 4, 6])
def test_every_potential_form(eng_mod, ptype):
    s = S.two_species_generic(ptype)
    o = _oracle(s)
    xyz = o.make_sites()
    ref = o.force_calc(xyz)
    e = eng_mod.ForceEngine(s)
    got = e.force_calc(s.h, xyz)
    assert rel_err(got["force"], ref["force"]) < TOL64
    assert abs(got["pe"] - ref["pe"]) <= TOL64 * abs(ref["pe"])
    # the same with no Ewald sum (kernel.c:356-461 forms)
    s.control.alpha = -1.0
    o = _oracle(s)
    ref = o.force_calc(xyz)
    e2 = eng_mod.ForceEngine(s)
    got = e2.force_calc(s.h, xyz)
    assert rel_err(got["force"], ref["force"]) < TOL64
    assert abs(got["pe"] - ref["pe"]) <= TOL64 * abs(ref["pe"])
    e.close()
    e2.close()


def test_clay_static_energy_matches_moldy_log(eng_mod):
    """The logged static clay run (step 0): real -5068.5, recip -4508.4 kJ/mol."""
    from moldy_amd import units
    s, exp = S.example("clay")
    e = eng_mod.ForceEngine(s)
    got = e.eval_forces()
    assert abs(got["pe"][0] * units.CONV_E - exp["pe_real_kjmol"]) < 0.06
    assert abs(got["pe"][1] * units.CONV_E - exp["pe_recip_kjmol"]) < 0.06
    e.close()


def test_force_calc_accumulates(eng_mod):
    """Callee accumulates into site_force/pe/stress (src/force.c:1114-1115)."""
    s = S.water(n=64)
    o = _oracle(s)
    xyz = o.make_sites()
    rng = np.random.default_rng(0)
    f0 = rng.normal(size=(3, s.nsites))
    ref = o.force_calc(xyz, f0.copy())
    e = eng_mod.ForceEngine(s)
    got = e.force_calc(s.h, xyz, f0.copy())
    assert rel_err(got["force"], ref["force"]) < TOL64
    assert rel_err(np.triu(got["stress"]), np.triu(ref["stress"])) < TOL64
    e.close()


@pytest.mark.parametrize("mode", [1, 2, 4])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("case", ["water", "salt", "silica", "mgclh2o", "argon"])
def test_overlapped_real_space_is_bitwise_serial(eng_mod, case, precision, mode):
    """The real-space pass on its own stream beside the Ewald sum sums every
    site force in the serial order: identical results either way."""
    s = CASES[case]()
    out = []
    for overlap in (False, True):
        e = eng_mod.ForceEngine(s, precision=precision)
        e.set_realspace_mode(mode)
        e.set_overlap(overlap)
        e.upload_state()
        for _ in range(2):
            pe, dip, st = e.eval_forces_device()
        out.append((pe.copy(), st.copy()) + tuple(x.copy() for x in e.download()))
        e.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("mode", [1, 2, 4])
@pytest.mark.parametrize("precision", [0, 1])
def test_too_close_pairs(eng_mod, precision, mode):
    """A hydrogen of one water 0.4 A from the oxygen of another: Moldy warns
    once for the pair (src/force.c:939-949, TOOCLS).  The engine reports the
    same count and the same pair of sites, from either real-space kernel and
    at either precision, and the FP64 forces still match."""
    s = S.close_pair_water()
    o = _oracle(s)
    xyz = o.make_sites()
    ref = o.force_calc(xyz)
    n = ref["info"].n_too_close
    assert n == 1
    want = {tuple(sorted((ref["info"].too_close_i[k], ref["info"].too_close_j[k]))) for k in range(n)}
    e = eng_mod.ForceEngine(s, precision=precision)
    e.set_realspace_mode(mode)
    got = e.force_calc(s.h, xyz)
    info = got["info"]
    assert info.n_too_close == n
    assert {tuple(sorted((info.too_close_i[k], info.too_close_j[k]))) for k in range(n)} == want
    if precision == 0:
        assert rel_err(got["force"], ref["force"]) < TOL64
        assert abs(got["pe"] - ref["pe"]) <= TOL64 * abs(ref["pe"])
    e.close()
