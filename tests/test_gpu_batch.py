"""Replicas stepped together (mgpu_batch_*) against each replica stepped on
its own (mgpu_md_steps): every schedule gives bit-identical trajectories,
since each replica runs the same kernels in the same order on its own
stream, or, grouped, the same blocks of the same kernels inside one launch
per stage.  The autotuner returns a valid schedule and shapes whose results
stay within rounding of the defaults."""
import numpy as np
import pytest

from moldy_amd import system

pytestmark = pytest.mark.gpu


def _replicas(precision, reps=None):
    from moldy_amd import engine as E
    reps = reps or system.water_replicas(nrep=5, seed=4, nmin=64, nmax=216)
    out = []
    for k, (s, T) in enumerate(reps):
        e = E.ForceEngine(s, precision=precision)
        e.set_dynamics(system.Dynamics(step=0.0005))
        e.upload_state()
        e.upload_momenta(*s.thermal_momenta(T, seed=k))
        out.append(e)
    return reps, out


def _check_against_single(precision, schedule, make):
    from moldy_amd import engine as E
    reps, single = _replicas(precision, make())
    ref = [e.md_steps(6, init_H_0=True, use_graph=False)[0] for e in single]
    ref_state = [e.download_dynamics() for e in single]
    ref2 = [e.md_steps(3, init_H_0=False, use_graph=False)[0] for e in single]
    ref2_state = [e.download_dynamics() for e in single]
    for e in single:
        e.close()
    reps, eng = _replicas(precision, make())
    b = E.Batch(eng)
    tr = b.steps(6, init_H_0=True, schedule=schedule)
    for r, e in enumerate(eng):
        assert np.array_equal(tr[r], ref[r]), r
        d = e.download_dynamics()
        for k in ("c_of_m", "quat", "mom", "amom"):
            assert np.array_equal(d[k], ref_state[r][k]), (r, k)
    # a second call replays the captured step from its first step on
    # (graph and grouped schedules): the same bits again
    tr2 = b.steps(3, schedule=schedule)
    for r, e in enumerate(eng):
        assert np.array_equal(tr2[r], ref2[r]), r
        d = e.download_dynamics()
        for k in ("c_of_m", "quat", "mom", "amom"):
            assert np.array_equal(d[k], ref2_state[r][k]), (r, k)
    b.close()
    for e in eng:
        e.close()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("schedule", [0, 1, 2, 3])
def test_batch_matches_single_replicas(precision, schedule):
    from moldy_amd import engine as E
    if precision == E.FP64 and schedule == E.SCHED_GROUPED:
        # the FP64 Ewald sum has no grouped launches: refused before any step
        reps, eng = _replicas(precision)
        before = [e.download_dynamics()["c_of_m"].copy() for e in eng]
        b = E.Batch(eng)
        with pytest.raises(E.EngineError):
            b.steps(2, schedule=schedule)
        for e, c in zip(eng, before):
            assert np.array_equal(e.download_dynamics()["c_of_m"], c)
        b.close()
        for e in eng:
            e.close()
        return
    _check_against_single(precision, schedule,
                          lambda: system.water_replicas(nrep=5, seed=4, nmin=64, nmax=216))


def test_grouped_uneven_replicas():
    """Grouped launches over replicas whose steps differ: a box large enough
    for the load-balanced real-space kernel beside small ones that take the
    shell-walk kernel, and k-space cutoffs that need different numbers of
    16-column blocks in the MFMA Ewald kernels."""
    from moldy_amd import engine as E

    def make():
        small = system.water_replicas(nrep=2, seed=7, nmin=40, nmax=120)
        large = system.water_replicas(nrep=1, seed=8, nmin=1500, nmax=1600)
        return [small[0], large[0], small[1]]
    _check_against_single(E.MIXED, E.SCHED_GROUPED, make)


def test_grouped_plan_launches():
    """One launch per stage: a grouped step makes about as many launches as
    one replica's step (a few more where the replicas' kernels differ), not
    the replicas' sum."""
    from moldy_amd import engine as E
    reps, eng = _replicas(E.MIXED)
    b = E.Batch(eng)
    with pytest.raises(E.EngineError):
        b.grouped_plan()              # not built yet
    b.steps(3, schedule=E.SCHED_GROUPED)
    g, own = b.grouped_plan()
    per = own / len(eng)
    print("grouped launches per step", g, "replica launches per step", own)
    assert per <= g <= 2 * per and g < own
    b.close()
    for e in eng:
        e.close()


def test_autotune():
    from moldy_amd import engine as E
    reps, eng = _replicas(1)
    before = [e.eval_forces_device()[0].copy() for e in eng]
    shapes = [e.autotune() for e in eng]
    after = [e.eval_forces_device()[0] for e in eng]
    for x, y in zip(before, after):
        assert np.allclose(x, y, rtol=1e-6, atol=0)
    b = E.Batch(eng)
    sched, ms = b.autotune(trial_steps=3)
    print("shapes", shapes, "schedule", E.SCHED_NAMES[sched], "ms/step", ms)
    assert sched in (0, 1, 2, 3) and np.all(ms > 0)
    tr = b.steps(4, init_H_0=True)
    assert np.all(np.isfinite(tr))
    b.close()
    for e in eng:
        e.close()


def test_autotune_beside_the_gridded_sum():
    """The gridded sum has no shapes to tune; a system of the same k rows and size
    class on the direct side of the size rule is tuned by itself, not given the
    shapes of one that never ran them."""
    from moldy_amd import engine as E, system
    s = system.water_box(2700, seed=3)          # 10,800 sites, 8.2e7 products: gridded
    d = s.copy()
    d.species = [system.water_species(2500)]    # 7.6e7: direct, the same box
    d.c_of_m, d.quat = s.c_of_m[:2500].copy(), s.quat[:2500].copy()
    assert s.nsites // 4096 == d.nsites // 4096
    out = []
    for x in (s, d):
        e = E.ForceEngine(x)
        e.upload_state()
        e.profile(True)
        pe = e.eval_forces_device()[0].copy()
        grid = e.profile_get("ewald_grid_spread")[1] > 0
        shape = e.autotune()
        assert np.allclose(e.eval_forces_device()[0], pe, rtol=1e-12, atol=0)
        out.append((grid, shape))
        e.close()
    assert out[0] == (True, (0, 0))
    assert out[1][0] is False and out[1][1][0] == 0 and out[1][1][1] in (4, 8, 16, 32)
