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
