"""Which sort the split replay beyond the LDS form uses, each against the oracle's sequential loop
(pyvibdmc.py:340-356): candidates ordered in LDS, or moved in global memory where a bucket of the
LDS order holds more than 64 of them, or where they are more than 31 744."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KILLS = dict(ordered=[4000, 6000, 6000, 6000], crowded=[4000, 6000, 6000, 6000], many=[4000, 30000, 30000, 30000])
WALKERS = dict(ordered=60_000, crowded=60_000, many=300_000)


def weights(kind, thresh=0.01, seed=5):
    """Weights of which about KILLS[kind][t] cross the threshold in step t.

    The potential is all but zero, so a step multiplies all weights by exp(-(W - N) / 2N), W their
    sum, which splits do not change: the groups are placed where the product of those factors takes
    them below.  `crowded`: the heaviest are a clump of distinct mantissas in 110 / 16384 of an octave,
    and twelve walkers heavier still whose mantissas span it, so that the clump falls into some 110 of
    the sort's buckets: up to 82 each in step 0, up to 177 in step 1 (a Python model of the key's map).
    Otherwise they are spread over an octave and more: at most 25 a bucket."""
    rs = np.random.RandomState(seed)
    n, kills = WALKERS[kind], KILLS[kind]
    heavy = np.empty(0)
    spread = 0.5
    if kind == 'crowded':
        clump = 4.0 * (1.5 + (110 / 16384) * rs.rand(9000)) / 1.5
        heavy = np.concatenate([clump, 16.0 * (1 + np.arange(12) / 12 + 0.01 * rs.rand(12))])
        spread = 0.02
    rest = np.exp(rs.uniform(-spread, spread, n - sum(kills) - len(heavy)))
    total, fallen, low = 1.15 * n, 0.0, []
    w = total
    for k in kills:
        d = 0.5 * (w - n) / n
        low.append(thresh * np.exp(fallen + d * rs.uniform(0.05, 0.95, k)))
        fallen, w = fallen + d, w * np.exp(-d)
    low = np.concatenate(low)
    rest *= (total - low.sum() - heavy.sum()) / rest.sum()
    out = np.concatenate([low, heavy, rest])
    rs.shuffle(out)
    return out


@pytest.mark.timeout(300)
@pytest.mark.parametrize('kind,ordered,moved', [('ordered', 3, 0), ('crowded', 0, 1), ('many', 0, 2)])
def test_replay_sorts_match_oracle(kind, ordered, moved):
    """Four steps of injected draws, FP64; the first has no candidate lists.  `ordered` and `moved` are
    the least counts of the two sorts.  Splits, weights and coordinates match (the weights are products
    of exp() factors: 1e-12)."""
    import pyvibdmc_amd as pv
    from oracle import pes as P
    from oracle.dmc import LegacyDraws, OracleDMC
    from pyvibdmc_amd import _native as N
    n, k = WALKERS[kind], 1e-5  # V dt about 5e-7: tells the walkers' weights apart, moves them by no more
    kw = dict(start_structures=np.random.RandomState(1).normal(0, 0.1, (n, 1, 3)), num_walkers=n,
              num_timesteps=4, delta_t=10, equil_steps=10 ** 9, wfn_every=10 ** 9, weighting='continuous',
              cont_wt_thresh=0.01, start_cont_wts=weights(kind))
    orc = OracleDMC(potential=lambda cds: P.harmonic_x(cds, k), masses=[P.M_H], draws=LegacyDraws(n % 100 + 3), **kw)
    orc.propagate()
    sim = pv.DMC_Sim(atoms=['X'], masses=P.M_H, potential=pv.HarmonicOscillator1D(k=k), precision='fp64',
                     rng=LegacyDraws(n % 100 + 3), write_files=False, chkpt_every=10 ** 9, **kw)
    sim.propagate()
    nb, how = sim.trajectory_counts(0, 4)
    c = (ctypes.c_int64 * 5)()
    N.check(N.load().pvd_sim_counts(sim._h, c, N.stream_handle()))
    print('splits', nb, 'replay', how, 'ordered', c[3], 'moved', c[4], flush=True)
    np.testing.assert_array_equal(nb, orc.rec['n_branched'])
    np.testing.assert_allclose(sim._vref_vs_tau, orc._vref_vs_tau, rtol=0, atol=1e-10)
    coords, wts = sim._get_walkers()
    np.testing.assert_array_equal(coords, orc.coords)
    np.testing.assert_allclose(wts, orc.cont_wts, rtol=1e-12, atol=0)
    assert how[0] == 2 and np.isin(how[1:], [7, 8]).all()
    assert c[3] >= ordered and c[4] >= moved and c[3] + c[4] == 3
