"""The parameter adjoint (mgpu_adjoint) against central finite differences of
the FP64 forward (h = 1e-6 relative), for every potential form and for the
charges: dE/dtheta, the cotangent product sum_i v_i . dF_i/dtheta and the
directional derivative of the site forces.  A torch.autograd.Function over
the C ABI (test harness only) gives the force-matching gradient, checked the
same way."""
import numpy as np
import pytest

import systems_small as S
from moldy_amd import system

pytestmark = pytest.mark.gpu

H_REL = 1e-6
TOL = 2e-6


def _cases():
    return {
        "silica": lambda: S.silica(),
        "water": lambda: S.water(n=64, cutoff=6.0),
        "salt": lambda: S.salt(),
        "argon": lambda: S.argon(),
        "mcy": lambda: S.two_species_generic(2, n=60),
        "generic": lambda: S.two_species_generic(3, n=60),
        "hiw": lambda: S.two_species_generic(4, n=60),
        "morse": lambda: S.two_species_generic(6, n=60),
    }


class Forward:
    """E and site forces of eval_forces at a given theta (FP64)."""

    def __init__(self, s):
        from moldy_amd import engine as E
        self.E = E
        self.s = s
        self.eng = E.ForceEngine(s)

    def __call__(self, theta):
        s2 = self.E.set_theta(self.s, theta)
        self.eng.rebind(s2)
        self.eng.upload_state()
        pe, _, _ = self.eng.eval_forces_device()
        _, _, _, sf = self.eng.download()
        return pe.sum(), sf

    def adjoint(self, theta, v=None, dtheta=None):
        s2 = self.E.set_theta(self.s, theta)
        self.eng.rebind(s2)
        self.eng.upload_state()
        return self.eng.adjoint(v=v, dtheta=dtheta)


def _steps(theta):
    # 1e-6 relative; parameters that are zero (pair types without that term,
    # uncharged ids) enter linearly or quadratically, where any step is exact
    return np.where(theta != 0.0, H_REL * np.abs(theta), 1e-2)


@pytest.mark.parametrize("case", list(_cases()))
def test_adjoint_vs_central_differences(case):
    from moldy_amd import engine as E
    s = _cases()[case]()
    fw = Forward(s)
    th = E.get_theta(s)
    rng = np.random.Generator(np.random.Philox(17))
    v = rng.standard_normal((3, s.nsites))
    dth = rng.standard_normal(th.size) * np.abs(th)
    got = fw.adjoint(th, v=v, dtheta=dth)
    h = _steps(th)
    fd_e = np.zeros(th.size)
    fd_v = np.zeros(th.size)
    for t in range(th.size):
        tp, tm = th.copy(), th.copy()
        tp[t] += h[t]
        tm[t] -= h[t]
        (ep, fp), (em, fm) = fw(tp), fw(tm)
        fd_e[t] = (ep - em) / (2 * h[t])
        fd_v[t] = (v * (fp - fm)).sum() / (2 * h[t])
    eps = 1e-6
    (_, fp), (_, fm) = fw(th + eps * dth), fw(th - eps * dth)
    fd_j = (fp - fm) / (2 * eps)
    ee = np.abs(got["dE"] - fd_e).max() / np.abs(fd_e).max()
    ev = np.abs(got["vjp"] - fd_v).max() / np.abs(fd_v).max()
    ej = np.linalg.norm(got["jvp"] - fd_j) / np.linalg.norm(fd_j)
    print(f"{case}: ntheta {th.size}  dE {ee:.1e}  vjp {ev:.1e}  jvp {ej:.1e}")
    assert ee < TOL and ev < TOL and ej < TOL
    fw.eng.close()


@pytest.mark.parametrize("case,subcell", [("argon", 8.5), ("argon", 0.9), ("water", 6.0), ("silica", 3.3), ("large", 0.0)])
def test_adjoint_occupancies(case, subcell):
    """Cells of many sites (a lane lists its cell in several rounds), of few
    (most lanes of a round list none), and a system whose waves take more
    than one site each; dE/dtheta and the cotangent product against central
    differences, the directional derivative against their pairing
    (v . jvp(dtheta) = dtheta . vjp(v)), which is exact in real arithmetic:
    FP64 sums of at most 1e7 terms, 1e-10."""
    from moldy_amd import engine as E
    if case == "large":
        s = system.argon_fcc(ncell=17, jitter=0.05, cutoff=6.0)
    else:
        s = _cases()[case]()
    s.control.subcell = subcell
    fw = Forward(s)
    th = E.get_theta(s)
    rng = np.random.Generator(np.random.Philox(23))
    v = rng.standard_normal((3, s.nsites))
    dth = rng.standard_normal(th.size) * np.abs(th)
    got = fw.adjoint(th, v=v, dtheta=dth)
    assert abs((v * got["jvp"]).sum() - dth @ got["vjp"]) < 1e-10 * np.abs(dth * got["vjp"]).sum()
    alone = fw.adjoint(th)           # no cotangent: the dE half only
    assert np.array_equal(alone["dE"], got["dE"])
    h = _steps(th)
    for t in np.flatnonzero(th)[:4]:
        tp, tm = th.copy(), th.copy()
        tp[t] += h[t]
        tm[t] -= h[t]
        (ep, fp), (em, fm) = fw(tp), fw(tm)
        assert abs((ep - em) / (2 * h[t]) - got["dE"][t]) < TOL * np.abs(got["dE"]).max()
        assert abs((v * (fp - fm)).sum() / (2 * h[t]) - got["vjp"][t]) < TOL * np.abs(got["vjp"]).max()
    fw.eng.close()


def test_force_matching_gradient_through_autograd():
    """Silica-like crystal, Buckingham: loss = |F(theta) - F_target|^2 with
    the target forces of a perturbed parameter set."""
    import torch
    from moldy_amd import engine as E
    s = S.silica()
    fw = Forward(s)
    th0 = E.get_theta(s)
    rng = np.random.Generator(np.random.Philox(5))
    th_true = th0 * (1 + 0.02 * rng.standard_normal(th0.size))
    _, F_target = fw(th_true)

    class SiteForces(torch.autograd.Function):
        @staticmethod
        def forward(ctx, theta):
            t = theta.detach().cpu().numpy()
            ctx.theta = t
            return torch.from_numpy(fw(t)[1])

        @staticmethod
        def backward(ctx, g):
            out = fw.adjoint(ctx.theta, v=g.detach().cpu().numpy().astype(np.float64))
            return torch.from_numpy(out["vjp"])

    theta = torch.tensor(th0, dtype=torch.float64, requires_grad=True)
    target = torch.from_numpy(F_target)
    loss = ((SiteForces.apply(theta) - target) ** 2).sum()
    loss.backward()
    g = theta.grad.numpy()
    h = _steps(th0)
    fd = np.zeros(th0.size)
    for t in range(th0.size):
        tp, tm = th0.copy(), th0.copy()
        tp[t] += h[t]
        tm[t] -= h[t]
        fd[t] = (((fw(tp)[1] - F_target) ** 2).sum() - ((fw(tm)[1] - F_target) ** 2).sum()) / (2 * h[t])
    err = np.abs(g - fd).max() / np.abs(fd).max()
    print(f"force matching: |grad| {np.abs(fd).max():.3e}  rel err {err:.1e}")
    assert err < TOL
    fw.eng.close()


def test_sixteen_ids():
    """Ten more ids without sites (the most an engine takes): every derivative as
    without them, zeros for theirs."""
    from moldy_amd import engine as E, system
    s = S.salt()
    n = 16
    big = s.copy()
    big.potpar = system.empty_potpar(n)
    big.potpar[:s.max_id, :s.max_id] = s.potpar
    big.site_mass = np.concatenate([s.site_mass, np.zeros(n - len(s.site_mass))])
    big.site_charge = np.concatenate([s.site_charge, np.zeros(n - s.max_id)])
    assert big.max_id == n
    npar = s.n_potpar
    pairs = [(a, b) for a in range(n) for b in range(a, n)]
    old = [(a, b) for a in range(s.max_id) for b in range(a, s.max_id)]
    at = [pairs.index(p) * npar + k for p in old for k in range(npar)]
    at += [len(pairs) * npar + a for a in range(s.max_id)]
    rng = np.random.default_rng(4)
    v = rng.standard_normal((3, s.nsites))
    th = E.get_theta(s)
    d = rng.standard_normal(th.size) * np.abs(th)
    dbig = np.zeros(E.get_theta(big).size)
    dbig[at] = d
    out = []
    for x, dt in ((s, d), (big, dbig)):
        e = E.ForceEngine(x)
        e.upload_state()
        out.append(e.adjoint(v=v, dtheta=dt))
        e.close()
    a, b = out
    rest = np.setdiff1d(np.arange(dbig.size), at)
    for k in ("dE", "vjp"):
        # sums over the waves' sites, cut differently: few eps of their terms
        assert np.linalg.norm(b[k][at] - a[k]) <= 1e-11 * np.linalg.norm(a[k])
        q = slice(-s.max_id, None)
        assert np.allclose(b[k][at][q], a[k][q], rtol=1e-9, atol=1e-11 * np.abs(a[k][q]).max())
        assert np.all(b[k][rest] == 0.0)
    assert np.linalg.norm(b["jvp"] - a["jvp"]) <= 1e-11 * np.linalg.norm(a["jvp"])
