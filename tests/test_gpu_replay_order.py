"""The split replay's two sorts beyond the LDS form: candidates ordered in LDS (up to 31 744) and
moved in global memory (more of them, or crowded buckets), against the oracle's sequential loop
(pyvibdmc.py:340-356)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.timeout(300)
@pytest.mark.parametrize('n,share,width', [
    (250_000, 0.25, 0.1),    # a few thousand kills: about the least that leave the LDS form
    (700_000, 0.45, 0.12),   # lists on both sides of what the LDS order holds
    (400_000, 0.30, 1e-3),   # every heavy walker in a band of a thousandth: crowded buckets
])
def test_replay_orders_match_oracle(n, share, width):
    """Four steps of injected draws, FP64: a share of the walkers just above the threshold (they
    cross it), the rest log-uniform over two e-folds, or over `width` where that is small.  Splits
    per step, weights and coordinates match (the weights are products of exp() factors: 1e-12)."""
    import pyvibdmc_amd as pv
    from oracle import pes as P
    from oracle.dmc import LegacyDraws, OracleDMC
    rs = np.random.RandomState(n % 1000 + 7)
    start = P.water_eq()[None] + rs.normal(0, 0.05, (n, 3, 3))
    w0 = np.exp(rs.uniform(-1.0, 1.0, n) if width > 0.01 else rs.uniform(0.0, width, n))
    band = rs.rand(n) < share
    w0[band] = 0.01 * np.exp(rs.uniform(0.0, max(width, 0.1), int(band.sum())))
    w0[~band] *= (n - w0[band].sum()) / w0[~band].sum()
    kw = dict(masses=[1837.15, 1837.15, 29156.95], start_structures=start, num_walkers=n, num_timesteps=4, delta_t=5,
              equil_steps=10 ** 9, wfn_every=10 ** 9, weighting='continuous', cont_wt_thresh=0.01, start_cont_wts=w0)
    orc = OracleDMC(potential=P.morse_bend, draws=LegacyDraws(n % 100 + 3), **kw)
    orc.propagate()
    sim = pv.DMC_Sim(atoms=['H', 'H', 'O'], potential=pv.MorseBendTriatomic(), precision='fp64',
                     rng=LegacyDraws(n % 100 + 3), write_files=False, chkpt_every=10 ** 9, **kw)
    sim.propagate()
    nb, how = sim.trajectory_counts(0, 4)
    print('splits', nb, 'replay', how, flush=True)
    np.testing.assert_array_equal(nb, orc.rec['n_branched'])
    np.testing.assert_allclose(sim._vref_vs_tau, orc._vref_vs_tau, rtol=0, atol=1e-10)
    coords, wts = sim._get_walkers()
    np.testing.assert_array_equal(coords, orc.coords)
    np.testing.assert_allclose(wts, orc.cont_wts, rtol=1e-12, atol=0)
