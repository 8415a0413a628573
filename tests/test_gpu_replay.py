"""Runs whose first step is a replay of the captured step (H_0 set by the
device's flag), against eager runs: bit-identical, over repeated calls, a call
longer than the one that captured the step, and a changed integrator step; and
uploads that return before their transfer, with the caller's arrays
overwritten at once."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _engine(prec, nvt):
    from moldy_amd import engine as E, system
    s = system.water_box(125, seed=21, cutoff=6.5, alpha=0.40)
    e = E.ForceEngine(s, precision=prec)
    e.set_dynamics(system.Dynamics(step=0.001, temp=300.0 if nvt else 0.0, const_temp=int(nvt)))
    return s, e


def _run(s, e, n, graph, init=True):
    mom, amom = s.thermal_momenta(300.0, seed=4)
    cm, q = s.c_of_m.copy(), s.quat.copy()
    e.upload_state(c_of_m=cm, quat=q)
    e.upload_momenta(mom, amom)
    for a in (cm, q, mom, amom):
        a[...] = 1e30      # the upload has taken its copy
    tr, pe, st = e.md_steps(n, init_H_0=init, use_graph=graph)
    d = e.download_dynamics()
    return [tr, pe, st, d["c_of_m"], d["quat"], d["mom"], d["amom"], np.array([d["ts"], d["tsmom"], d["H_0"]])]


@pytest.mark.parametrize("nvt", [False, True])
@pytest.mark.parametrize("prec", [0, 1])
def test_replayed_first_step_is_bitwise_eager(prec, nvt):
    from moldy_amd import system
    s, e = _engine(prec, nvt)
    for n in (3, 3, 1, 7, 2):
        a, b = _run(s, e, n, True), _run(s, e, n, False)
        assert all(np.array_equal(x, y) for x, y in zip(a, b))
        assert np.all(np.isfinite(a[0])) and a[0][0, 6] != 0.0
    # H_0 is kept when not asked for
    assert np.array_equal(_run(s, e, 2, True, init=False)[0][:, 6], np.zeros(2))
    e.set_dynamics(system.Dynamics(step=0.0005, temp=300.0 if nvt else 0.0, const_temp=int(nvt)))
    a, b = _run(s, e, 4, True), _run(s, e, 4, False)
    assert all(np.array_equal(x, y) for x, y in zip(a, b))
    e.close()


def test_profile_times_the_first_step_of_every_call():
    """With profiling on, a call's first step runs eagerly with its timing events
    although the captured step is current; the same bits."""
    from moldy_amd import engine as E
    s, e = _engine(1, False)
    want = _run(s, e, 4, True)
    e.profile(True)
    for calls in (1, 2):
        got = _run(s, e, 4, True)
        assert all(np.array_equal(x, y) for x, y in zip(got, want))
        assert e.profile_get("realspace")[1] == calls
    b = E.Batch([e])
    for schedule in (E.SCHED_GRAPH, E.SCHED_GROUPED):
        for _ in range(2):
            e.profile(True)
            e.upload_state()
            e.upload_momenta(*s.thermal_momenta(300.0, seed=4))
            tr = b.steps(4, init_H_0=True, schedule=schedule)
            assert np.array_equal(tr[0], want[0])
            assert e.profile_get("realspace")[1] == 1
    b.close()
    e.profile(False)
    assert np.array_equal(_run(s, e, 4, True)[0], want[0])
    e.close()


def test_upload_without_a_buffer_is_an_error():
    """Missing arrays are refused with a status (the copy into pinned memory
    would read them), and the engine goes on as it was."""
    import ctypes as C
    from moldy_amd import engine as E, system
    s = system.water_box(64, seed=21, cutoff=5.5, alpha=0.40)
    e = E.ForceEngine(s)
    want = e.eval_forces()
    L, dp = E.lib(), C.POINTER(C.c_double)
    h, cm, q = (np.ascontiguousarray(x, np.float64) for x in (s.h, s.c_of_m, s.quat))
    p = [x.ctypes.data_as(dp) for x in (h, cm, q)]
    for missing in range(3):
        args = [None if k == missing else p[k] for k in range(3)]
        assert L.mgpu_upload_state(e.h_, *args) == 1      # MGPU_E_ARG
        assert b"bad buffers" in L.mgpu_last_error(e.h_)
    pe, dip, st = e.eval_forces_device()
    assert np.array_equal(pe, want["pe"]) and np.array_equal(st, want["stress"])
    # atoms have no quaternions to give
    a = system.argon_fcc(4, cutoff=8.5)
    ea = E.ForceEngine(a)
    h, cm = np.ascontiguousarray(a.h), np.ascontiguousarray(a.c_of_m)
    assert L.mgpu_upload_state(ea.h_, h.ctypes.data_as(dp), cm.ctypes.data_as(dp), None) == 0
    ea.eval_forces_device()
    e.close()
    ea.close()


def test_replay_after_another_precision():
    """A captured mixed step, an FP64 evaluation (other tables of the gridded
    reciprocal sum), then the mixed run again: the capture is not reused with
    the other precision's tables."""
    from moldy_amd import engine as E, system
    s = system.water_box(5000, seed=23)
    e = E.ForceEngine(s, precision=E.MIXED)
    e.set_dynamics(system.Dynamics(step=0.001, temp=0.0, const_temp=0))
    a = _run(s, e, 3, True)
    e.set_precision(E.FP64)
    e.upload_state()
    e.eval_forces_device()
    e.set_precision(E.MIXED)
    b = _run(s, e, 3, True)
    c = _run(s, e, 3, False)
    assert all(np.array_equal(x, y) for x, y in zip(a, b))
    assert all(np.array_equal(x, y) for x, y in zip(a, c))
    e.close()
