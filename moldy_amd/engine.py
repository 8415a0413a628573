"""ctypes front end of libmoldy_amd.so (the C ABI in include/moldy_amd.h).

``ForceEngine`` mirrors the reference's operator interface for this path:
``force_calc`` and ``ewald`` take site coordinates and accumulate into site
forces, energy and the upper-triangle virial exactly like src/force.c:1108
and src/ewald.c:280; ``eval_forces`` is the device-resident restatement of
src/accel.c:398-617.  The library is required: importing this module on a
machine where it was not built raises.
"""
import ctypes as C
import os

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
LIBPATH = os.path.join(HERE, "libmoldy_amd.so")

FP64, MIXED = 0, 1
_dp = C.POINTER(C.c_double)
_ip = C.POINTER(C.c_int)
_lp = C.POINTER(C.c_long)

ERRORS = {1: "ARG", 2: "HIP", 3: "BIN_RANGE", 4: "BIN_ROUND", 5: "CUTOFF", 6: "TONAB",
          7: "MULTIFW", 8: "PTYPE", 9: "STATE", 10: "CAPACITY", 11: "QNORM"}
TRACE_W = 8


class EngineError(RuntimeError):
    def __init__(self, code, msg):
        super().__init__(f"mgpu error {code} ({ERRORS.get(code, '?')}): {msg}")
        self.code = code


class MgpuSystem(C.Structure):
    _fields_ = [("nsites", C.c_int), ("nmols", C.c_int), ("nspecies", C.c_int),
                ("max_id", C.c_int), ("ptype", C.c_int), ("n_potpar", C.c_int),
                ("spec_nmols", _ip), ("spec_nsites", _ip), ("spec_framework", _ip),
                ("spec_rdof", _ip), ("spec_site_id", _ip), ("spec_p_f_sites", _dp),
                ("site_charge", _dp), ("potpar", _dp),
                ("cutoff", C.c_double), ("subcell", C.c_double), ("alpha", C.c_double),
                ("k_cutoff", C.c_double), ("strict_cutoff", C.c_int), ("molpbc", C.c_int),
                ("surface_dipole", C.c_int)]


class FcInfo(C.Structure):
    _fields_ = [("nx", C.c_int), ("ny", C.c_int), ("nz", C.c_int), ("n_nabors", C.c_int),
                ("n_too_close", C.c_int), ("too_close_i", C.c_int * 16),
                ("too_close_j", C.c_int * 16), ("n_list_entries", C.c_long),
                ("max_cell_sites", C.c_int), ("eintra", C.c_double)]


class MgpuDynamics(C.Structure):
    _fields_ = [("step", C.c_double), ("ttmass", C.c_double), ("pmass", C.c_double),
                ("gkt", C.c_double), ("const_temp", C.c_int), ("nosymmetric_rot", C.c_int),
                ("spec_mass", _dp), ("spec_inertia", _dp), ("const_pressure", C.c_int),
                ("pressure", C.c_double), ("strain_mask", C.c_int)]


class EwInfo(C.Structure):
    _fields_ = [("hmax", C.c_int), ("kmax", C.c_int), ("lmax", C.c_int), ("nhkl", C.c_int),
                ("nsitesxf", C.c_int), ("self_energy", C.c_double),
                ("sheet_energy", C.c_double)]


_LIB = None


def lib():
    global _LIB
    if _LIB is None:
        if not os.path.exists(LIBPATH):
            raise ImportError(f"{LIBPATH} is not built; run `python -m moldy_amd.build`")
        L = C.CDLL(LIBPATH)
        L.mgpu_last_error.restype = C.c_char_p
        L.mgpu_last_error.argtypes = [C.c_void_p]
        L.mgpu_destroy.argtypes = [C.c_void_p]
        _LIB = L
    return _LIB


def _p(a, t=_dp):
    return a.ctypes.data_as(t) if a is not None else None


def get_theta(system):
    """theta of the parameter adjoint: the n_potpar parameters of each
    site-id pair a <= b (row order over 0..max_id-1), then the charges."""
    m, npar = system.max_id, system.n_potpar
    out = []
    for a in range(m):
        for b in range(a, m):
            out.extend(system.potpar[a, b, :npar])
    out.extend(system.site_charge)
    return np.array(out, np.float64)


def set_theta(system, theta):
    """A copy of system with theta's parameters and charges."""
    s = system.copy()
    m, npar = s.max_id, s.n_potpar
    q = 0
    for a in range(m):
        for b in range(a, m):
            s.potpar[a, b, :npar] = theta[q:q + npar]
            s.potpar[b, a, :npar] = theta[q:q + npar]
            q += npar
    s.site_charge[:] = theta[q:q + m]
    return s


SCHED_GRAPH, SCHED_STREAM_GRAPHS, SCHED_STREAMS, SCHED_GROUPED = 0, 1, 2, 3
SCHED_NAMES = ["graph", "stream_graphs", "streams", "grouped"]


class Batch:
    """Replicas stepped together (mgpu_batch_*): engines prepared for MD."""

    def __init__(self, engines, device=0):
        L = lib()
        L.mgpu_batch_last_error.restype = C.c_char_p
        L.mgpu_batch_last_error.argtypes = [C.c_void_p]
        L.mgpu_batch_destroy.argtypes = [C.c_void_p]
        b = C.c_void_p()
        rc = L.mgpu_batch_create(C.byref(b), int(device))
        if rc:
            raise EngineError(rc, "mgpu_batch_create")
        self.b = b
        self.engines = list(engines)
        for e in self.engines:
            self._chk(L.mgpu_batch_add(self.b, e.h_))

    def _chk(self, rc):
        if rc:
            raise EngineError(rc, lib().mgpu_batch_last_error(self.b).decode())

    def steps(self, nsteps, init_H_0=False, schedule=-1):
        """Returns trace[n_replicas][nsteps][8] (mgpu_md_steps layout)."""
        tr = np.zeros((len(self.engines), max(nsteps, 1), TRACE_W))
        self._chk(lib().mgpu_batch_steps(self.b, int(nsteps), int(init_H_0), int(schedule), _p(tr)))
        return tr[:, :nsteps]

    def grouped_plan(self):
        """(launches per step of the grouped schedule, the replicas' own
        launches per step summed), once the grouped schedule has run."""
        out = (C.c_long * 2)()
        self._chk(lib().mgpu_batch_grouped_plan(self.b, out))
        return int(out[0]), int(out[1])

    def autotune(self, trial_steps=4):
        """(schedule, ms per step of each schedule; -1 where one does not apply)."""
        s = C.c_int()
        ms = np.zeros(len(SCHED_NAMES))
        self._chk(lib().mgpu_batch_autotune(self.b, int(trial_steps), C.byref(s), _p(ms)))
        return s.value, ms

    def close(self):
        if getattr(self, "b", None):
            lib().mgpu_batch_destroy(self.b)
            self.b = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


class ForceEngine:
    """One engine (HIP stream + device buffers) bound to one system."""

    def __init__(self, system, device=0, precision=FP64):
        L = lib()
        h = C.c_void_p()
        self._chk(L.mgpu_create(C.byref(h), int(device)), h)
        self.h_ = h
        self.rebind(system)
        self.set_precision(precision)

    def rebind(self, system):
        """(Re)describe the system to the engine (mgpu_set_system); the state
        must be uploaded again afterwards."""
        L = lib()
        self.sys = system
        self.f = system.flat()
        f, c = self.f, system.control
        self.cs = MgpuSystem(system.nsites, system.nmols, system.nspecies, system.max_id,
                             system.ptype, system.n_potpar,
                             _p(f["spec_nmols"], _ip), _p(f["spec_nsites"], _ip),
                             _p(f["spec_framework"], _ip), _p(f["spec_rdof"], _ip),
                             _p(f["spec_site_id"], _ip), _p(f["spec_p_f_sites"]),
                             _p(f["site_charge"]), _p(f["potpar"]),
                             c.cutoff, c.subcell, c.alpha, c.k_cutoff, int(c.strict_cutoff),
                             int(c.molpbc), int(c.surface_dipole))
        self._chk(L.mgpu_set_system(self.h_, C.byref(self.cs)))
        self.chg = system.site_charges()

    def _chk(self, rc, h=None):
        if rc:
            hh = h if h is not None else self.h_
            msg = lib().mgpu_last_error(hh).decode() if hh else ""
            raise EngineError(rc, msg)

    def close(self):
        if getattr(self, "h_", None):
            lib().mgpu_destroy(self.h_)
            self.h_ = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def set_precision(self, p):
        self._chk(lib().mgpu_set_precision(self.h_, int(p)))
        self.precision = p

    def set_overlap(self, on):
        """Real-space pass on a second stream beside the Ewald sum."""
        self._chk(lib().mgpu_set_overlap(self.h_, int(bool(on))))

    RS_AUTO, RS_WALK, RS_BALANCED, RS_BALANCED_SEARCH, RS_TILED = 0, 1, 2, 3, 4

    def set_realspace_mode(self, mode):
        """Real-space kernel: RS_AUTO, RS_WALK (per-offset walk),
        RS_BALANCED (waves over the sites, candidates from the shell's
        z-columns), RS_BALANCED_SEARCH (the same, candidates placed in
        windows of 64 instead of 2048) or
        RS_TILED (Newton-3: every pair once, one block per z-column of cells,
        half of the shell's columns staged in LDS)."""
        self._chk(lib().mgpu_set_realspace_mode(self.h_, int(mode)))

    def realspace_balanced(self):
        """Whether the last real-space pass used a column kernel (2, 3, 4)."""
        return bool(lib().mgpu_realspace_balanced(self.h_))

    # ------------------------------------------------------- the boundary
    def force_calc(self, h, xyz, fxyz=None, chg=None, c_of_m=None):
        n = self.sys.nsites
        xyz = np.ascontiguousarray(xyz, np.float64)
        f = np.zeros((3, n)) if fxyz is None else fxyz
        pe = C.c_double(0.0)
        st = np.zeros(9)
        info = FcInfo()
        h = np.ascontiguousarray(h, np.float64)
        cm = np.ascontiguousarray(self.sys.c_of_m if c_of_m is None else c_of_m, np.float64)
        q = np.ascontiguousarray(self.chg if chg is None else chg, np.float64)
        self._chk(lib().mgpu_force_calc(self.h_, _p(h), _p(xyz), n, _p(cm), _p(q), _p(f),
                                        C.byref(pe), _p(st), C.byref(info)))
        return dict(force=f, pe=pe.value, stress=st.reshape(3, 3), info=info)

    def ewald(self, h, xyz, fxyz=None, chg=None):
        n = self.sys.nsites
        xyz = np.ascontiguousarray(xyz, np.float64)
        f = np.zeros((3, n)) if fxyz is None else fxyz
        pe = C.c_double(0.0)
        st = np.zeros(9)
        info = EwInfo()
        h = np.ascontiguousarray(h, np.float64)
        q = np.ascontiguousarray(self.chg if chg is None else chg, np.float64)
        self._chk(lib().mgpu_ewald(self.h_, _p(h), _p(xyz), n, _p(q), _p(f), C.byref(pe),
                                   _p(st), C.byref(info)))
        return dict(force=f, pe=pe.value, stress=st.reshape(3, 3), info=info)

    # --------------------------------------------------- device resident
    def upload_state(self, h=None, c_of_m=None, quat=None):
        s = self.sys
        h = np.ascontiguousarray(s.h if h is None else h, np.float64)
        cm = np.ascontiguousarray(s.c_of_m if c_of_m is None else c_of_m, np.float64)
        q = np.ascontiguousarray(self.f["quat"] if quat is None else quat, np.float64)
        self._chk(lib().mgpu_upload_state(self.h_, _p(h), _p(cm), _p(q)))

    def eval_forces_device(self):
        pe = np.zeros(2)
        dip = np.zeros(3)
        st = np.zeros(9)
        self._chk(lib().mgpu_eval_forces(self.h_, _p(pe), _p(dip), _p(st)))
        return pe, dip, st.reshape(3, 3)

    def download(self):
        s = self.sys
        force = np.zeros((s.nmols, 3))
        torque = np.zeros((max(s.nmols_r, 1), 3))
        sx = np.zeros((3, s.nsites))
        sf = np.zeros((3, s.nsites))
        self._chk(lib().mgpu_download_forces(self.h_, _p(force), _p(torque), _p(sx), _p(sf)))
        return force, torque[:s.nmols_r], sx, sf

    def eval_forces(self, h=None, c_of_m=None, quat=None):
        self.upload_state(h, c_of_m, quat)
        pe, dip, st = self.eval_forces_device()
        force, torque, sx, sf = self.download()
        return dict(pe=pe, dip=dip, stress=st, force=force, torque=torque, site_xyz=sx,
                    site_force=sf)

    def last_info(self):
        fc, ew = FcInfo(), EwInfo()
        lib().mgpu_last_info(self.h_, C.byref(fc), C.byref(ew))
        return fc, ew

    # -------------------------------------------------- molecular dynamics
    def set_dynamics(self, dyn):
        """dyn: moldy_amd.system.Dynamics (program units)."""
        from moldy_amd import units
        s = self.sys
        mass, inertia = s.species_mass_inertia()
        self._dyn_arrays = (np.ascontiguousarray(mass), np.ascontiguousarray(inertia))
        self.dyn = MgpuDynamics(dyn.step, dyn.ttmass, dyn.pmass,
                                s.degrees_of_freedom() * units.KB * dyn.temp,
                                int(dyn.const_temp), int(dyn.nosymmetric_rot),
                                _p(self._dyn_arrays[0]), _p(self._dyn_arrays[1]),
                                int(dyn.const_pressure), float(dyn.pressure), int(dyn.strain_mask))
        self._chk(lib().mgpu_set_dynamics(self.h_, C.byref(self.dyn)))

    def upload_momenta(self, mom, amom, ts=1.0, tsmom=0.0, H_0=0.0):
        mom = np.ascontiguousarray(mom, np.float64)
        amom = np.ascontiguousarray(amom, np.float64)
        th = np.array([ts, tsmom, H_0])
        self._chk(lib().mgpu_upload_momenta(self.h_, _p(mom), _p(amom), _p(th)))

    def md_steps(self, nsteps, init_H_0=False, use_graph=True):
        """Runs nsteps do_steps; returns (trace[nsteps][8], pe[2], stress[3,3])."""
        tr = np.zeros((max(nsteps, 1), TRACE_W))
        pe = np.zeros(2)
        st = np.zeros(9)
        self._chk(lib().mgpu_md_steps(self.h_, int(nsteps), int(init_H_0), int(use_graph),
                                      _p(tr), _p(pe), _p(st)))
        return tr[:nsteps], pe, st.reshape(3, 3)

    def download_dynamics(self):
        s = self.sys
        cm = np.zeros((s.nmols, 3))
        q = np.zeros((max(s.nmols_r, 1), 4))
        mom = np.zeros((s.nmols, 3))
        amom = np.zeros((max(s.nmols_r, 1), 4))
        th = np.zeros(3)
        self._chk(lib().mgpu_download_dynamics(self.h_, _p(cm), _p(q), _p(mom), _p(amom), _p(th)))
        return dict(c_of_m=cm, quat=q[:s.nmols_r], mom=mom, amom=amom[:s.nmols_r], ts=th[0],
                    tsmom=th[1], H_0=th[2])

    def upload_cell_momentum(self, hmom):
        hm = np.ascontiguousarray(hmom, np.float64).reshape(9)
        self._chk(lib().mgpu_upload_cell_momentum(self.h_, _p(hm)))

    def download_cell(self):
        """(h, hmom) as 3x3 arrays: the cell after the last run."""
        h, hm = np.zeros(9), np.zeros(9)
        self._chk(lib().mgpu_download_cell(self.h_, _p(h), _p(hm)))
        return h.reshape(3, 3), hm.reshape(3, 3)

    # ------------------------------------------------ cells and pair lists
    def cells(self, h, xyz, c_of_m=None):
        s = self.sys
        xyz = np.ascontiguousarray(xyz, np.float64)
        h = np.ascontiguousarray(h, np.float64)
        cm = np.ascontiguousarray(s.c_of_m if c_of_m is None else c_of_m, np.float64)
        dims = np.zeros(3, np.int32)
        self._chk(lib().mgpu_cells(self.h_, _p(h), _p(xyz), s.nsites, _p(cm), _p(dims, _ip),
                                   None, None, None))
        nc = int(np.prod(dims))
        ne = s.nsites if not s.control.molpbc else None
        ne = self._nentries()
        ec = np.zeros(ne, np.int32)
        cs = np.zeros(nc + 1, np.int32)
        ce = np.zeros(ne, np.int32)
        self._chk(lib().mgpu_cells(self.h_, _p(h), _p(xyz), s.nsites, _p(cm), _p(dims, _ip),
                                   _p(ec, _ip), _p(cs, _ip), _p(ce, _ip)))
        return dict(dims=tuple(dims), entry_cell=ec, cell_start=cs, cell_entries=ce)

    def _nentries(self):
        s = self.sys
        if not s.control.molpbc:
            return s.nsites
        return sum(sp.nmols * (sp.nsites if sp.framework else 1) for sp in s.species)

    def pairlist(self, h, xyz, strict=None, cutoff=None, c_of_m=None):
        s = self.sys
        c = s.control
        xyz = np.ascontiguousarray(xyz, np.float64)
        h = np.ascontiguousarray(h, np.float64)
        cm = np.ascontiguousarray(s.c_of_m if c_of_m is None else c_of_m, np.float64)
        strict = int(c.strict_cutoff if strict is None else strict)
        cut = c.cutoff if cutoff is None else cutoff
        dims = self.cells(h, xyz, cm)["dims"]
        nc = int(np.prod(dims))
        total = C.c_long()
        starts = np.zeros(nc + 1, np.int64)
        self._chk(lib().mgpu_pairlist(self.h_, _p(h), _p(xyz), s.nsites, _p(cm), strict,
                                      C.c_double(cut), C.byref(total), _p(starts, _lp),
                                      None, None, None))
        n = total.value
        nab = np.zeros(n + 1, np.int32)
        pbc = np.zeros(n + 1, np.int32)
        nf = np.zeros((nc, 2), np.int32)
        self._chk(lib().mgpu_pairlist(self.h_, _p(h), _p(xyz), s.nsites, _p(cm), strict,
                                      C.c_double(cut), C.byref(total), _p(starts, _lp),
                                      _p(nab, _ip), _p(pbc, _ip), _p(nf, _ip)))
        return dict(start=starts, nab=nab[:n], pbctrans=pbc[:n], nfnab=nf)

    def autotune(self, reps=3):
        """Launch shapes by timing (mgpu_autotune): (sk_blocks, npart)."""
        a, b = C.c_int(), C.c_int()
        self._chk(lib().mgpu_autotune(self.h_, int(reps), C.byref(a), C.byref(b)))
        return a.value, b.value

    # ------------------------------------------------- parameter adjoint
    def theta_count(self):
        n = C.c_int()
        self._chk(lib().mgpu_theta_count(self.h_, C.byref(n)))
        return n.value

    def adjoint(self, v=None, dtheta=None, want_dE=True):
        """dE/dtheta, sum_i v_i . dF_i/dtheta and sum_t dtheta_t dF/dtheta_t
        at the uploaded state (theta layout: get_theta)."""
        nt = self.theta_count()
        ns = self.sys.nsites
        dE = np.zeros(nt) if want_dE else None
        vj = np.zeros(nt) if v is not None else None
        jv = np.zeros((3, ns)) if dtheta is not None else None
        vv = np.ascontiguousarray(v, np.float64) if v is not None else None
        dt = np.ascontiguousarray(dtheta, np.float64) if dtheta is not None else None
        self._chk(lib().mgpu_adjoint(self.h_, _p(vv), _p(dt), _p(dE), _p(vj), _p(jv)))
        return dict(dE=dE, vjp=vj, jvp=jv)

    # ------------------------------------------ radial distribution functions
    def rdf(self, h, xyz, limit, nbins, rdf=None, c_of_m=None):
        """rdf_inner/rdf_accum on the GPU: float bins [(max_id-1)*max_id/2][nbins],
        accumulated into ``rdf`` when given."""
        s = self.sys
        nblk = (s.max_id - 1) * s.max_id // 2
        out = np.zeros((nblk, nbins), np.float32) if rdf is None else rdf
        assert out.dtype == np.float32 and out.flags.c_contiguous and out.size == nblk * nbins
        xyz = np.ascontiguousarray(xyz, np.float64)
        h = np.ascontiguousarray(h, np.float64)
        cm = np.ascontiguousarray(s.c_of_m if c_of_m is None else c_of_m, np.float64)
        self._chk(lib().mgpu_rdf(self.h_, _p(h), _p(xyz), s.nsites, _p(cm), C.c_double(limit),
                                 int(nbins), out.ctypes.data_as(C.POINTER(C.c_float))))
        return out

    # --------------------------------------------------------- profiling
    def profile(self, on=True):
        lib().mgpu_profile_enable(self.h_, int(on))
        lib().mgpu_profile_reset(self.h_)

    def profile_get(self, name):
        ms = C.c_double()
        n = C.c_long()
        lib().mgpu_profile_get(self.h_, name.encode(), C.byref(ms), C.byref(n))
        return ms.value, n.value

    def sync(self):
        self._chk(lib().mgpu_sync(self.h_))
