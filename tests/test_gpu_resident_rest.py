"""Discrete steps of a launch that was given up because its workgroups could not all run at once:
the workgroups of a second launch that do run take them, one or all.  They follow the same shares and
the same sums, so every result equals the undisturbed run's bit for bit, vref included.  A gate wait
of zero gives every launch up."""
import ctypes

import numpy as np
import pytest

from tests.test_gpu_resident import drive, make

pytestmark = pytest.mark.gpu


def counts(sim):
    """Launches with the walkers on chip, launches given up, redistributions."""
    from pyvibdmc_amd import _native as N
    c = (ctypes.c_int64 * 5)()
    N.check(N.load().pvd_sim_counts(sim._h, c, N.stream_handle()))
    return list(c)[:3]


def waits(sim, gate, team):
    from pyvibdmc_amd import _native as N
    N.check(N.load().pvd_sim_resident_waits(sim._h, gate, team))


def equal(a, b):
    assert a['rc'] == b['rc'] and a['fail_step'] == b['fail_step']
    for k in ('pop', 'counts', 'walkers', 'eff', 'vref', 'final'):
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)
    for k in a.get('wfn', {}):
        np.testing.assert_array_equal(a['wfn'][k], b['wfn'][k], err_msg=k)


FORMS = [
    ('ho', 'fp64', 257, 120, None, {}),            # two workgroups
    ('ho', 'fp32', 5000, 200, 100, {}),
    ('water', 'fp32', 100003, 240, 120, {}),       # with redistributions
    ('water', 'fp64', 30011, 130, None, {}),
    ('water', 'fp32', 300_000, 150, None, {}),     # several rounds a workgroup
    ('water', 'fp32', 30000, 120, None, dict(branch_every=3)),
    ('ps', 'fp32', 20000, 100, None, {}),
    ('cluster', 'fp32', 60000, 120, 60, {}),
    ('water', 'fp32', 100003, 130, None, dict(imp_samp='water_trial')),
    ('ps', 'fp32', 20000, 100, None, dict(imp_samp='water_trial')),
    ('cluster', 'fp32', 60001, 120, None, dict(imp_samp='cluster6_trial')),
    ('water', 'fp32', 20000, 120, None, dict(imp_samp='water_trial', branch_every=3)),
    ('water', 'fp32', 20000, 200, None, dict(DEBUG_alpha=-0.5)),   # fails on the way
    ('water', 'fp32', 20000, 200, None, dict(DEBUG_alpha=-0.5, imp_samp='water_trial')),
]


@pytest.mark.parametrize('system,precision,n,steps,window,kw', FORMS)
def test_given_up_launches_match_undisturbed(system, precision, n, steps, window, kw):
    import pyvibdmc_amd as pv
    runs = []
    for gate, team in ((-1, -1), (0, -1), (0, 0)):  # undisturbed; all workgroups late; the first few alone
        kw2 = dict(kw, imp_samp=getattr(pv, kw['imp_samp'])()) if 'imp_samp' in kw else kw
        sim = make(system, n, steps, precision, **kw2)
        waits(sim, gate, team)
        runs.append(drive(sim, steps, False, window))
        o, c, _ = counts(sim)
        assert (c == 0 and o > 0) if gate < 0 else (o == 0 and c > 0), (o, c)
    for r in runs[1:]:
        equal(runs[0], r)
    if 'DEBUG_alpha' in kw:
        assert runs[0]['rc'] != 0 and runs[0]['fail_step'] > 2


def test_given_up_launches_between_others():
    """Launches given up and not, and single launches, in turn within one run."""
    from pyvibdmc_amd import _native as N
    got = []
    for disturbed in (False, True):
        sim = make('water', 50000, 400, 'fp32')
        sim._start()
        for i, m in enumerate((100, 3, 120, 1, 110)):
            waits(sim, 0 if disturbed and i == 2 else -1, -1)
            N.check(N.load().pvd_sim_run(sim._h, m, N.stream_handle()))
        rc, _, _ = sim._status()
        assert rc == 0
        sim._fetch_traj(0, 334)
        got.append((sim._pop_vs_tau[:334].copy(), sim._vref_vs_tau[:334].copy(), sim._get_walkers()[0], counts(sim)[:2]))
    for a, b in zip(got[0][:3], got[1][:3]):
        np.testing.assert_array_equal(a, b)
    assert got[0][3] == [3, 0] and got[1][3] == [2, 1]
