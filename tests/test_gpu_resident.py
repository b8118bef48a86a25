"""Discrete steps with the walkers kept on chip (many steps per launch) against the same steps
launched one at a time: the draws and the per-walker arithmetic are the same, so populations,
births, deaths, descendant weights and walkers agree bit for bit; vref is a sum over the walkers
in another order (FP64, fewer than 2^21 terms of one magnitude: 1e-12 relative is ample)."""
import numpy as np
import pytest

from oracle import pes as P

pytestmark = pytest.mark.gpu


def make(system, n, steps, precision, **kw):
    import pyvibdmc_amd as pv
    rs = np.random.RandomState(n % 1000)
    common = dict(num_walkers=n, num_timesteps=steps, precision=precision, seed=11, write_files=False,
                  equil_steps=10 ** 9, wfn_every=10 ** 9, chkpt_every=10 ** 9)
    if system == 'ho':
        common.update(atoms=['X'], masses=P.M_H, delta_t=10,
                      potential=pv.HarmonicOscillator1D(k=P.M_H * P.HO_OMEGA ** 2),
                      start_structures=rs.normal(0, 0.1, (n, 1, 3)))
    elif system == 'cluster':
        common.update(atoms=['O', 'H', 'H', 'O', 'H', 'H'], masses=[P.M_O, P.M_H, P.M_H, P.M_O, P.M_H, P.M_H],
                      delta_t=5, potential=pv.TwoMonomerCluster(),
                      start_structures=P.cluster6_eq()[None] + rs.normal(0, 0.05, (n, 6, 3)))
    else:
        pot = pv.PartridgeSchwenkeWater() if system == 'ps' else pv.MorseBendTriatomic()
        common.update(atoms=['H', 'H', 'O'], masses=[P.M_H, P.M_H, P.M_O], delta_t=5, potential=pot,
                      start_structures=P.water_eq()[None] + rs.normal(0, 0.05, (n, 3, 3)))
    common.update(kw)
    return pv.DMC_Sim(**common)


def drive(sim, steps, one_by_one, window=None):
    """Run `steps` steps in one call, or one call per step (the launch-per-step kernels);
    `window`: descendant tracking from that step on."""
    from pyvibdmc_amd import _native as N
    lib, st = N.load(), N.stream_handle()
    sim._start()
    legs = [steps] if window is None else [window, steps - window]
    for leg, m in enumerate(legs):
        if leg == 1:
            N.check(lib.pvd_sim_desc_begin(sim._h, st))
        for k in ([1] * m if one_by_one else [m]):
            N.check(lib.pvd_sim_run(sim._h, k, st))
    rc, status, fail_step = sim._status()
    out = dict(rc=rc, fail_step=fail_step)
    done = steps if rc == 0 else fail_step
    sim._fetch_traj(0, steps)
    out.update(pop=sim._pop_vs_tau[:done].copy(), vref=sim._vref_vs_tau[:done].copy(), walkers=sim._get_walkers()[0],
               counts=np.stack(sim.trajectory_counts(0, steps))[:, :done],
               eff=None if sim.eff_ts is None else sim.eff_ts[:done].copy(), final=sim._vref)
    if window is not None:
        sim._save_wfn(window)
        out['wfn'] = sim.wfns[-1][1]
    return out


def same(a, b):
    assert a['rc'] == b['rc'] and a['fail_step'] == b['fail_step']
    for k in ('pop', 'counts', 'walkers', 'eff'):
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)
    np.testing.assert_allclose(a['vref'], b['vref'], rtol=1e-12, atol=0)
    np.testing.assert_allclose(a['final'], b['final'], rtol=1e-12, atol=0)
    if 'wfn' in a:
        for k in a['wfn']:
            np.testing.assert_array_equal(a['wfn'][k], b['wfn'][k], err_msg=k)


@pytest.mark.parametrize('system,precision,n,steps,window', [
    ('ho', 'fp64', 60, 40, None),            # one partly filled wave
    ('ho', 'fp64', 5000, 100, 60),
    ('ho', 'fp32', 257, 40, None),           # two workgroups
    ('water', 'fp32', 16, 20, None),
    ('water', 'fp32', 65536, 70, None),      # every workgroup exactly one round
    ('water', 'fp32', 100003, 60, 30),
    ('water', 'fp32', 1_000_000, 60, 30),    # the LDS full, and with the tracker beyond it
    ('water', 'fp64', 70001, 40, None),
    ('water', 'fp64', 500_000, 40, None),
    ('ps', 'fp32', 20000, 40, None),
    ('ps', 'fp64', 5000, 30, None),
    ('cluster', 'fp32', 131_072, 60, 20),
    ('cluster', 'fp32', 499_979, 40, None),
])
def test_resident_steps_match_single_launches(system, precision, n, steps, window):
    runs = []
    for one in (False, True):
        sim = make(system, n, steps, precision)
        runs.append(drive(sim, steps, one, window))
        del sim
    assert runs[0]['rc'] == 0
    same(*runs)


@pytest.mark.parametrize('system,n,steps', [('water', 300, 40), ('water', 100003, 40), ('water', 1_000_000, 50),
                                            ('ps', 20000, 30), ('cluster', 499_979, 40)])
def test_resident_importance_sampling_matches_single_launches(system, n, steps):
    import pyvibdmc_amd as pv
    trial = pv.cluster6_trial if system == 'cluster' else pv.water_trial
    runs = [drive(make(system, n, steps, 'fp32', imp_samp=trial()), steps, one) for one in (False, True)]
    assert runs[0]['rc'] == 0
    same(*runs)


def test_resident_branch_every_matches_single_launches():
    import pyvibdmc_amd as pv
    for kw in ({}, dict(imp_samp=pv.water_trial())):
        same(*[drive(make('water', 30000, 40, 'fp32', branch_every=3, **kw), 40, one) for one in (False, True)])


@pytest.mark.parametrize('imp', [False, True])
def test_resident_failure_leaves_the_failed_steps_walkers(imp):
    """A run whose population leaves the guard after some steps: the same step, status and
    walkers as single launches (the on-chip walkers are retraced to the failed step)."""
    import pyvibdmc_amd as pv
    kw = dict(imp_samp=pv.water_trial()) if imp else {}
    runs = [drive(make('water', 20000, 200, 'fp32', DEBUG_alpha=-0.5, **kw), 200, one) for one in (False, True)]
    assert runs[0]['rc'] != 0 and runs[0]['fail_step'] > 2
    same(*runs)


def test_resident_steps_on_two_streams_from_two_threads():
    """Two simulations in two threads, each on its own stream: as run one after the other."""
    import threading
    import torch
    import pyvibdmc_amd as pv
    jobs = [('water', 100003, 'fp32', {}), ('water', 65536, 'fp32', dict(imp_samp=pv.water_trial()))]
    alone = [drive(make(s, n, 200, p, **kw), 200, False) for s, n, p, kw in jobs]
    got = [None, None]

    def work(i):
        s, n, p, kw = jobs[i]
        with torch.cuda.stream(torch.cuda.Stream()):
            got[i] = drive(make(s, n, 200, p, **kw), 200, False)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(alone, got):
        same(a, b)
