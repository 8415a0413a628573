"""Mixed precision (FP32 pair forces, split-FP16 MFMA Ewald, FP64 reductions)
against the FP64 path.  The accuracy bar of the mixed path: RMS relative
force error <= 1e-5; energies and stress are reported per quantity and held to the bounds
below."""
import numpy as np
import pytest

from conftest import rel_err
import systems_small as S
from test_gpu_parity import CASES

pytestmark = pytest.mark.gpu

TOL_F = 1e-5      # forces: the mixed path's accuracy bar
TOL_E = 3e-6      # reciprocal-space energy (1.1-1.4e-6 at the bench size and in skewed cells)
TOL_E_REAL = 1e-4 # real-space energy: FP32 pair energies of cancelling Coulomb terms
TOL_S = 3e-5      # stress: FP32 pair virials of ionic crystals cancel strongly (quartz 1.4e-5)


@pytest.mark.parametrize("case", [c for c in CASES if not c.startswith("argon")])
def test_mixed_ewald_vs_oracle(case):
    from moldy_amd import engine as E
    from oracle.oracle import Oracle
    s = CASES[case]()
    o = Oracle(s)
    xyz = o.make_sites()
    ref = o.ewald(xyz)
    e = E.ForceEngine(s, precision=E.MIXED)
    got = e.ewald(s.h, xyz)
    err_f = rel_err(got["force"], ref["force"])
    err_e = abs(got["pe"] - ref["pe"]) / abs(ref["pe"])
    print(f"{case}: recip force rms rel {err_f:.2e}  energy rel {err_e:.2e}")
    assert err_f < TOL_F
    assert err_e < TOL_E
    assert rel_err(np.triu(got["stress"]), np.triu(ref["stress"])) < TOL_E
    e.close()


@pytest.mark.parametrize("case", list(CASES))
def test_mixed_eval_vs_fp64(case):
    from moldy_amd import engine as E
    s = CASES[case]()
    e64 = E.ForceEngine(s, precision=E.FP64)
    r64 = e64.eval_forces()
    emx = E.ForceEngine(s, precision=E.MIXED)
    rmx = emx.eval_forces()
    errs = dict(site=rel_err(rmx["site_force"], r64["site_force"]),
                mol=rel_err(rmx["force"], r64["force"]),
                torque=rel_err(rmx["torque"], r64["torque"]) if s.nmols_r else 0.0,
                pe0=abs(rmx["pe"][0] - r64["pe"][0]) / abs(r64["pe"][0]),
                pe1=abs(rmx["pe"][1] - r64["pe"][1]) / max(abs(r64["pe"][1]), 1e-300),
                stress=rel_err(rmx["stress"], r64["stress"]))
    print(case, {k: f"{v:.2e}" for k, v in errs.items()})
    assert errs["site"] < TOL_F
    assert errs["mol"] < TOL_F
    assert errs["torque"] < TOL_F
    assert errs["pe0"] < TOL_E_REAL and errs["pe1"] < TOL_E
    assert errs["stress"] < TOL_S
    e64.close()
    emx.close()


def test_mixed_one_group_backprojection():
    """A box 20 times taller than wide: the k set reaches l = 58, so the MFMA
    back-projection runs with one group of waves (more than 48 columns); the
    mixed evaluation holds the same bar against FP64 as everywhere else."""
    from moldy_amd import engine as E
    s = S.tall_water()
    e64 = E.ForceEngine(s, precision=E.FP64)
    r64 = e64.eval_forces()
    emx = E.ForceEngine(s, precision=E.MIXED)
    rmx = emx.eval_forces()
    assert emx.last_info()[1].lmax >= 48
    err = rel_err(rmx["site_force"], r64["site_force"])
    print("tall water: site force rms rel", f"{err:.2e}")
    assert err < TOL_F
    assert rel_err(rmx["force"], r64["force"]) < TOL_F
    assert abs(rmx["pe"][1] - r64["pe"][1]) / abs(r64["pe"][1]) < TOL_E
    assert rel_err(rmx["stress"], r64["stress"]) < TOL_S
    e64.close()
    emx.close()


@pytest.mark.parametrize("name", ["water216", "water512", "water729", "salt900"])
def test_small_systems_keep_fp64_sums_of_pairs(name):
    """Below 16 sites a CU the balanced kernel sums FP32 pairs in FP64, as the
    walk does: the same error against FP64 to 0.5% (FP32 sums over a lane's pairs
    of a site were 1.6 to 2.3% off; all runs are deterministic).  The energy is a
    sum of 1e5 pairs whose rounding errors cancel at random: not compared."""
    from moldy_amd import engine as E, system
    s = (system.salt_water(nwater=900, nmg=16, ncl=32, seed=7) if name == "salt900"
         else system.water_box(int(name[5:]), seed=5))
    e = E.ForceEngine(s, precision=E.FP64)
    xyz = e.eval_forces()["site_xyz"]
    ref = e.force_calc(s.h, xyz)["force"]
    e.close()
    err = {}
    for mode in (E.ForceEngine.RS_AUTO, E.ForceEngine.RS_WALK):
        e = E.ForceEngine(s, precision=E.MIXED)
        e.set_realspace_mode(mode)
        err[mode] = rel_err(e.force_calc(s.h, xyz)["force"], ref)
        assert e.realspace_balanced() == (mode == E.ForceEngine.RS_AUTO)
        e.close()
    print(name, {k: f"{v:.4e}" for k, v in err.items()})
    assert err[E.ForceEngine.RS_AUTO] < 1.005 * err[E.ForceEngine.RS_WALK]
