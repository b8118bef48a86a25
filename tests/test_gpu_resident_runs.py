"""Runs long enough for the resident steps, in every form, against the same steps launched one at a
time: redistributions with and without the descendant tracker, launches in a row, a failure after a
redistribution, short legs in between.  The counts say that one side ran on chip and the other did
not."""
import numpy as np
import pytest

from tests.test_gpu_resident import drive, make, same
from tests.test_gpu_resident_rest import counts

pytestmark = pytest.mark.gpu


def pair(system, precision, n, steps, window, kw=None, spreads=None):
    """Both runs; the least number of redistributions on chip."""
    import pyvibdmc_amd as pv
    runs = []
    for one in (False, True):
        kw2 = dict(kw or {})
        if 'imp_samp' in kw2:
            kw2['imp_samp'] = getattr(pv, kw2['imp_samp'])()
        if kw2.get('potential'):
            kw2['potential'] = pv.HarmonicOscillator1D(k=kw2['potential'])
        sim = make(system, n, steps, precision, **kw2)
        runs.append(drive(sim, steps, one, window))
        c = counts(sim)
        print(system, precision, n, 'one by one' if one else 'together', c, runs[-1]['fail_step'])
        assert c == [0, 0, 0] if one else (c[0] > 0 and c[1] == 0)
        if spreads is not None and not one:
            assert c[2] >= spreads
    same(*runs)
    return runs


@pytest.mark.parametrize('system,precision,n,steps,window,spreads', [
    ('ho', 'fp64', 60, 200, 100, None),           # one workgroup
    ('ho', 'fp64', 5000, 250, 120, None),
    ('ho', 'fp32', 257, 200, None, None),
    ('ho', 'fp32', 1_000_000, 120, None, None),
    ('water', 'fp32', 65536, 200, 100, None),     # half of a round
    ('water', 'fp32', 122_880, 200, 100, 1),      # two rounds of 512 threads, in registers
    ('water', 'fp32', 100003, 300, 140, 1),
    ('water', 'fp32', 1_000_000, 240, 130, 1),    # the LDS full, and with the tracker beyond it
    ('water', 'fp64', 70001, 200, 100, None),
    ('water', 'fp64', 122_880, 200, 100, 1),
    ('water', 'fp64', 500_000, 120, None, 1),
    ('ps', 'fp32', 20000, 200, 100, None),
    ('ps', 'fp32', 300_000, 120, None, None),
    ('ps', 'fp64', 5000, 120, None, None),
    ('cluster', 'fp32', 131_072, 200, 100, None),
    ('cluster', 'fp32', 499_979, 120, None, None),
])
def test_runs_match_single_launches(system, precision, n, steps, window, spreads):
    assert pair(system, precision, n, steps, window, spreads=spreads)[0]['rc'] == 0


@pytest.mark.parametrize('precision,n', [('fp32', 5000), ('fp64', 300), ('fp32', 400_000)])
def test_one_component_matches_single_launches(precision, n):
    from oracle import pes as P
    kw = dict(potential=P.M_H * P.HO_OMEGA ** 2, start_structures=np.random.RandomState(3).normal(0, 0.1, (n, 1, 1)))
    assert pair('ho', precision, n, 200, 100, kw)[0]['rc'] == 0


@pytest.mark.parametrize('system,n,steps', [('water', 300, 200), ('water', 100003, 200), ('water', 1_000_000, 130),
                                            ('ps', 20000, 150), ('cluster', 60001, 200), ('cluster', 499_979, 120)])
def test_importance_sampled_runs_match_single_launches(system, n, steps):
    trial = 'cluster6_trial' if system == 'cluster' else 'water_trial'
    assert pair(system, 'fp32', n, steps, None, dict(imp_samp=trial))[0]['rc'] == 0


def test_launches_in_a_row_from_an_odd_step():
    """4 500 steps in one call, more than a launch takes, from step 97."""
    assert pair('water', 'fp32', 20000, 97 + 4500, 97, None)[0]['rc'] == 0


@pytest.mark.parametrize('n,kw', [(122_880, dict(DEBUG_alpha=-0.001)),
                                  (122_880, dict(DEBUG_alpha=-0.001, imp_samp='water_trial')),
                                  (480_000, dict(DEBUG_alpha=-0.0005))])  # with launches queued behind the failed one
def test_failure_after_a_redistribution(n, kw):
    """The retraced steps start from a redistribution, not from the launch's first step."""
    runs = pair('water', 'fp32', n, 3000, None, kw, spreads=1)
    assert runs[0]['rc'] != 0 and runs[0]['fail_step'] > 100


def test_short_legs_between():
    """On-chip legs, single launches and graphs in turn, with a window over them."""
    from pyvibdmc_amd import _native as N
    lib, got = N.load(), []
    for one in (False, True):
        sim, st = make('water', 50001, 600, 'fp32'), N.stream_handle()
        sim._start()
        for i, m in enumerate((70, 100, 3, 30, 1, 15, 200, 2, 64)):
            if i == 2:
                N.check(lib.pvd_sim_desc_begin(sim._h, st))
            for k in ([1] * m if one else [m]):
                N.check(lib.pvd_sim_run(sim._h, k, st))
            if i == 5:
                sim._status()
                sim._save_wfn(170)
        assert sim._status()[0] == 0
        sim._fetch_traj(0, 485)
        got.append(dict(pop=sim._pop_vs_tau[:485].copy(), vref=sim._vref_vs_tau[:485].copy(), rc=0, fail_step=-1,
                        walkers=sim._get_walkers()[0], counts=np.stack(sim.trajectory_counts(0, 485)), eff=None,
                        final=sim._vref, wfn=sim.wfns[-1][1]))
        assert counts(sim)[0] == (0 if one else 4)
    same(*got)


def test_first_steps_stay_with_the_step_kernels():
    """A run of a few steps does not pay for bringing the resident kernels to the device."""
    from pyvibdmc_amd import _native as N
    sim = make('water', 5000, 400, 'fp32')
    sim._start()
    for m, launches in ((5, 0), (20, 0), (70, 0), (15, 0), (16, 1), (200, 2)):
        N.check(N.load().pvd_sim_run(sim._h, m, N.stream_handle()))
        assert counts(sim)[0] == launches, m
    sim = make('water', 5000, 400, 'fp32')
    sim._start()
    N.check(N.load().pvd_sim_run(sim._h, 96, N.stream_handle()))
    assert counts(sim)[0] == 1
