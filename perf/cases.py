"""Timing cases of the package: what a user of it has it do, through its public entry points.

Three families:

* whole simulations: ``DMC_Sim(...)``, ``propagate()``, then the trajectory, the walkers and the
  saved wave functions, as a simulation script does it (host start structures in, host walkers
  out), in every weighting and propagation form and in both precisions;
* the learned potential on walkers that already live on the GPU: ``SurrogateModel.energy_planes``;
* one training step in its two calls: ``loss_and_grads`` (forward and backward) and ``adam_step``
  (update and repacking of the operands).

``listed()`` are fixed sizes, ``draw(rng)`` gives others of the same ranges.  ``prepare`` makes
inputs from the seed alone, ``run`` is one pass, ``exact`` the same numbers in 64 bits where a
closed evaluation exists (a stochastic trajectory has none).
"""
import math

import numpy as np
import torch

import pyvibdmc_amd as pv
from pyvibdmc_amd import _native as N
from pyvibdmc_amd.surrogate import SurrogatePotential

M_H, M_O = 1837.15, 29156.95
DE, A_M, RE, KB, TH0 = 0.1916, 1.2, 1.81, 0.16, math.radians(104.5)
CL = dict(De_oo=0.008, a_oo=0.8, re_oo=5.5, qO=-0.8, qH=0.4)
HO_OMEGA = 0.013669

# atoms, masses, equilibrium, sorting, nuclear charges of the two molecules
WATER_EQ = np.array([[RE, 0.0, 0.0], [RE * math.cos(TH0), RE * math.sin(TH0), 0.0], [0.0, 0.0, 0.0]])
_MONO = WATER_EQ[[2, 0, 1]]
CLUSTER_EQ = np.concatenate([_MONO, _MONO + np.array([0.0, 0.0, CL['re_oo']])])
MOLECULES = {
    'water': dict(el=['H', 'H', 'O'], mass=[M_H, M_H, M_O], eq=WATER_EQ, z=[1, 1, 8], atoms=[[0, 1], [2]], groups=None),
    'cluster': dict(el=['O', 'H', 'H', 'O', 'H', 'H'], mass=[M_O, M_H, M_H, M_O, M_H, M_H], eq=CLUSTER_EQ,
                    z=[8, 1, 1, 8, 1, 1], atoms=[[0], [1, 2], [3], [4, 5]], groups=[[0, 1, 2], [3, 4, 5]]),
}
NEVER = 10 ** 9


def listed():
    return [
        # the smallest ordinary run: a few thousand walkers of a model oscillator in double
        # precision, where a step is launches and latency
        dict(name='oscillator_5k_fp64', kind='sim', system='oscillator', form='plain', n=5000, steps=2000,
             precision='fp64', desc=False),
        # a production run of a small molecule, with descendant weighting (50 of every 500 steps)
        dict(name='water_100k', kind='sim', system='water', form='plain', n=100_000, steps=2000, precision='fp32',
             desc=True),
        # the large plain run (one million walkers)
        dict(name='water_1m', kind='sim', system='water', form='plain', n=1_000_000, steps=10_000, precision='fp32',
             desc=False),
        # importance sampling: drift, Metropolis and local energy of a Gaussian-product trial
        dict(name='water_is_1m', kind='sim', system='water', form='is', n=1_000_000, steps=4000, precision='fp32',
             desc=False),
        # importance sampling on the learned potential inside the step loop, an odd size
        dict(name='water_is_learned_400k', kind='sim', system='water', form='learned', n=400_003, steps=800,
             precision='fp32', desc=False),
        # continuous weighting with splitting of the heaviest walkers, with descendant weighting
        dict(name='water_continuous_100k', kind='sim', system='water', form='continuous', n=100_000, steps=1500,
             precision='fp32', desc=True),
        # the same where thousands of walkers are replaced on every step, in double precision
        dict(name='water_continuous_1m_fp64', kind='sim', system='water', form='continuous', n=1_000_000, steps=400,
             precision='fp64', desc=False),
        # a six-atom cluster with importance sampling, a ragged size
        dict(name='cluster_is_500k', kind='sim', system='cluster', form='is', n=499_979, steps=3000, precision='fp32',
             desc=False),
        # the cluster's network (15 -> 256 -> 256 -> 256 -> 1) on a million walkers, ragged
        dict(name='energy_256_1m', kind='energy', system='cluster', hidden=256, n=1_000_003, precision='fp32'),
        # forward and backward of a training step at the batch the training uses
        dict(name='grads_128_8192', kind='grads', system='water', hidden=128, n=8192),
        dict(name='grads_256_8192', kind='grads', system='cluster', hidden=256, n=8192),
        # the update that follows it: Adam and the repacked operands, the smallest call
        dict(name='adam_128', kind='adam', system='water', hidden=128),
    ]


def _log_size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(['sim', 'sim', 'sim', 'sim', 'energy', 'grads', 'grads', 'adam'])
    if kind == 'sim':
        system, form, top = rng.choice([('oscillator', 'plain', 1_000_000), ('water', 'plain', 1_000_000),
                                        ('water', 'is', 1_000_000), ('water', 'learned', 500_000),
                                        ('water', 'continuous', 1_000_000), ('cluster', 'plain', 500_000),
                                        ('cluster', 'is', 500_000)])
        precision = 'fp32' if form == 'learned' else rng.choice(['fp32', 'fp32', 'fp64'])
        if precision == 'fp64':
            top //= 2
        n = _log_size(rng, 2000, top)
        most = 400 if form == 'continuous' else 800 if form == 'learned' else 2000
        return dict(kind='sim', system=system, form=form, n=n, steps=rng.randint(most // 4, most),
                    precision=precision, desc=form in ('plain', 'continuous') and rng.random() < 0.3)
    system = rng.choice(['water', 'cluster'])
    hidden = rng.choice([128, 256])
    if kind == 'energy':
        return dict(kind='energy', system=system, hidden=hidden, n=_log_size(rng, 1000, 1_000_000),
                    precision=rng.choice(['fp32', 'fp32', 'fp64']))
    if kind == 'grads':
        return dict(kind='grads', system=system, hidden=hidden, n=_log_size(rng, 100, 20_000))
    return dict(kind='adam', system=system, hidden=hidden, seed_step=rng.randint(1, 50_000))


# ----------------------------------------------------------------- potentials in plain torch
def _morse_bend(h1, h2, o):
    u, v = h1 - o, h2 - o
    r1, r2 = u.norm(dim=-1), v.norm(dim=-1)
    th = torch.acos(((u * v).sum(-1) / (r1 * r2)).clamp(-1, 1))
    return DE * (1 - torch.exp(-A_M * (r1 - RE))) ** 2 + DE * (1 - torch.exp(-A_M * (r2 - RE))) ** 2 \
        + 0.5 * KB * (th - TH0) ** 2


def _potential(system, x):
    """V of (n, M, 3) walkers, in the type of x."""
    if system == 'water':
        return _morse_bend(x[:, 0], x[:, 1], x[:, 2])
    v = _morse_bend(x[:, 1], x[:, 2], x[:, 0]) + _morse_bend(x[:, 4], x[:, 5], x[:, 3])
    v = v + CL['De_oo'] * (1 - torch.exp(-CL['a_oo'] * ((x[:, 0] - x[:, 3]).norm(dim=-1) - CL['re_oo']))) ** 2
    q = [CL['qO'], CL['qH'], CL['qH']]
    for i in range(3):
        for j in range(3):
            v = v + q[i] * q[j] / (x[:, i] - x[:, 3 + j]).norm(dim=-1)
    return v


def _features(mol, x):
    """Inverse distances (n, D) of (n, M, 3) walkers after sorting like atoms, then groups, by
    the row norms of the Coulomb matrix, largest first."""
    n, m = x.shape[:2]
    z = torch.tensor(mol['z'], dtype=x.dtype, device=x.device)
    inv = 1.0 / ((x[:, :, None] - x[:, None]).norm(dim=-1) + torch.eye(m, dtype=x.dtype, device=x.device))
    inv = inv * (1 - torch.eye(m, dtype=x.dtype, device=x.device))
    norm = ((z[:, None] * z * inv) ** 2).sum(-1) + (0.5 * z ** 2.4) ** 2
    norm = norm.sqrt()
    order = torch.arange(m, device=x.device).repeat(n, 1)
    for sub in mol['atoms']:
        s = torch.tensor(sub, device=x.device)
        order[:, sub] = s[torch.argsort(norm[:, sub], dim=1, descending=True, stable=True)]
    if mol['groups']:
        g = torch.tensor(mol['groups'], device=x.device)
        tot = torch.gather(norm, 1, order)[:, g].sum(-1)
        to = torch.argsort(tot, dim=1, descending=True, stable=True)
        order = torch.gather(order, 1, g[to].reshape(n, -1))
    i, j = torch.triu_indices(m, m, 1)
    return inv[torch.arange(n, device=x.device)[:, None], order[:, i], order[:, j]]


# ------------------------------------------------------------------------------- the network
def _walkers(system, n, seed, spread):
    eq = MOLECULES[system]['eq']
    return eq[None] + np.random.RandomState(seed % (1 << 32)).normal(0.0, spread, (n,) + eq.shape)


_KNOWN = {}


def _description(system):
    """Normalisation, range and quadratic baseline of the network, fitted to the analytic surface
    on thermal geometries (plain numbers: what a finished training leaves in the description)."""
    if system not in _KNOWN:
        mol = MOLECULES[system]
        x = torch.from_numpy(_walkers(system, 32768, 77, 0.08))
        f = _features(mol, x).numpy()
        v = _potential(system, x).numpy()
        mean = f.mean(0).astype(np.float32)
        xinv = (1.0 / f.std(0)).astype(np.float32)
        xn = (f - mean) * xinv
        d = f.shape[1]
        cols = [np.ones(len(f))] + [xn[:, i] for i in range(d)]
        cols += [xn[:, i] * xn[:, j] for i in range(d) for j in range(i, d)]
        des = np.stack(cols, 1)
        quad = np.linalg.solve(des.T @ des + 1e-9 * np.eye(des.shape[1]), des.T @ v).astype(np.float32)
        res = v - des @ quad
        _KNOWN[system] = dict(mean=mean, xinv=xinv, lo=f.min(0).astype(np.float32), hi=f.max(0).astype(np.float32),
                              quad=quad, ymean=float(np.float32(res.mean())), ystd=float(np.float32(res.std())))
    return _KNOWN[system]


def _weights(system, hidden, seed):
    rs = np.random.RandomState((seed + 5) % (1 << 32))
    d = len(_description(system)['mean'])
    w = {}
    for k, (o, i) in enumerate([(hidden, d), (hidden, hidden), (hidden, hidden)]):
        w['W%d' % k] = (rs.uniform(-1, 1, (o, i)) * math.sqrt(6.0 / (i + o))).astype(np.float32)
        w['b%d' % k] = (rs.normal(0, 0.05, o)).astype(np.float32)
    w['w3'] = (rs.uniform(-1, 1, hidden) * math.sqrt(6.0 / (hidden + 1))).astype(np.float32)
    w['b3'] = rs.normal(0, 0.05, 1).astype(np.float32)
    return w


def _model(system, hidden, seed):
    mol, q = MOLECULES[system], _description(system)
    m = pv.SurrogateModel(mol['el'], hidden=hidden, sorted_atoms=mol['atoms'], sorted_groups=mol['groups'])
    for k in range(m.D):
        m.desc.xmean[k], m.desc.xinv[k] = float(q['mean'][k]), float(q['xinv'][k])
        m.desc.lo[k], m.desc.hi[k] = float(q['lo'][k]), float(q['hi'][k])
    for k, c in enumerate(q['quad']):
        m.desc.quad[k] = float(c)
    m.desc.ymean, m.desc.ystd = q['ymean'], q['ystd']
    m.set_params(_weights(system, hidden, seed))
    return m


def _network(w, x):
    """y (n) of normalised features x (n, D) in the type of x."""
    silu = torch.nn.functional.silu
    h = x
    for k in range(3):
        h = silu(h @ w['W%d' % k].t() + w['b%d' % k])
    return h @ w['w3'] + w['b3']


def _analytic(system):
    return pv.MorseBendTriatomic() if system == 'water' else pv.TwoMonomerCluster()


def _batch(system, n, seed):
    """Normalised features (D, n) and targets (n) of a training batch, on the GPU."""
    q = _description(system)
    x = torch.from_numpy(_walkers(system, n, seed, 0.08)).cuda()
    f = _features(MOLECULES[system], x)
    xt = ((f.float() - torch.from_numpy(q['mean']).cuda()) * torch.from_numpy(q['xinv']).cuda()).t().contiguous()
    xn = xt.t().double()
    d = xn.shape[1]
    cols = [torch.ones_like(xn[:, 0])] + [xn[:, i] for i in range(d)]
    cols += [xn[:, i] * xn[:, j] for i in range(d) for j in range(i, d)]
    base = torch.stack(cols, 1) @ torch.from_numpy(q['quad']).cuda().double()
    return xt, ((_potential(system, x) - base - q['ymean']) / q['ystd']).float()


# ------------------------------------------------------------------------------- the passes
def prepare(case, seed):
    kind, system = case['kind'], case['system']
    if kind == 'sim':
        return _prepare_sim(case, seed)
    if kind == 'energy':
        m = _model(system, case['hidden'], seed)
        m.desc.use_range = 1
        x = torch.from_numpy(_walkers(system, case['n'], seed, 0.08)).cuda()
        planes = x.reshape(case['n'], -1).t().contiguous()
        fp32 = case['precision'] == 'fp32'
        return dict(kind=kind, model=m, planes=planes.float().contiguous() if fp32 else planes,
                    out=torch.empty(case['n'], dtype=torch.float64, device='cuda'),
                    precision=N.PVD_FP32 if fp32 else N.PVD_FP64, fallback=_analytic(system))
    m = _model(system, case['hidden'], seed)
    if kind == 'grads':
        xt, t = _batch(system, case['n'], seed)
        return dict(kind=kind, model=m, x=xt, t=t)
    # adam: a training under way (moments of earlier steps)
    g = torch.Generator().manual_seed(seed % (1 << 62))
    k = m.params.numel()
    m.grads.copy_(1e-3 * torch.randn(k, generator=g))
    m.m1.copy_(1e-3 * torch.randn(k, generator=g))
    m.m2.copy_(1e-6 * torch.rand(k, generator=g))
    m.t = int(case.get('seed_step', 1000))
    return dict(kind=kind, model=m)


def _prepare_sim(case, seed):
    system, form, n = case['system'], case['form'], case['n']
    rs = np.random.RandomState(seed % (1 << 32))
    kw = dict(num_walkers=n, num_timesteps=case['steps'], precision=case['precision'], rng='philox', seed=int(seed),
              write_files=False, chkpt_every=NEVER)
    kw.update(equil_steps=500, wfn_every=500, desc_wt_steps=50) if case['desc'] else \
        kw.update(equil_steps=NEVER, wfn_every=NEVER)
    if system == 'oscillator':
        kw.update(atoms=['X'], masses=M_H, delta_t=10, potential=pv.HarmonicOscillator1D(k=M_H * HO_OMEGA ** 2),
                  start_structures=rs.normal(0.0, 0.1, (n, 1, 3)))
        return dict(kind='sim', kw=kw, kept={})
    mol = MOLECULES[system]
    kw.update(atoms=mol['el'], masses=mol['mass'], delta_t=5, potential=_analytic(system),
              start_structures=mol['eq'][None] + rs.normal(0.0, 0.05, (n,) + mol['eq'].shape))
    if form in ('is', 'learned'):
        kw['imp_samp'] = pv.water_trial() if system == 'water' else pv.cluster6_trial()
    if form == 'learned':
        kw['potential'] = SurrogatePotential(_model(system, 128, seed), _analytic(system), judge_every=100)
    if form == 'continuous':
        kw.update(weighting='continuous', cont_wt_thresh=0.01)
    return dict(kind='sim', kw=kw, kept={})


def _keep(state, key, rows):
    """Rows of a population into the program's own array of the largest population allowed (the
    rest zero), so that results of runs with different populations line up."""
    most = max(len(rows), int(1.5 * state['kw']['num_walkers']) + 1)
    buf, used = state['kept'].get(key, (None, 0))
    if buf is None:
        buf = np.zeros((most,) + rows.shape[1:])
    buf[:len(rows)] = rows
    buf[len(rows):used] = 0.0
    state['kept'][key] = (buf, len(rows))
    return buf


def run(state):
    kind = state['kind']
    if kind == 'sim':
        sim = pv.DMC_Sim(**state['kw'])
        sim.propagate()
        coords, wts = sim.walkers if sim.weighting == 'continuous' else (sim.walkers, None)
        return dict(vref=sim.vref_vs_tau, population=len(coords), walkers=_keep(state, 'walkers', coords), weights=wts,
                    wfns=[{k: _keep(state, (t, k), v) for k, v in rec.items()} for t, rec in getattr(sim, 'wfns', [])])
    m = state['model']
    if kind == 'energy':
        p = state['planes']
        m.energy_planes(p.data_ptr(), p.shape[1], None, p.shape[1], state['out'], state['precision'],
                        state['fallback'])
        return state['out']
    if kind == 'grads':
        loss, y = m.loss_and_grads(state['x'], state['t'])
        return dict(loss=loss, y=y, grads=m.grads)
    m.adam_step(1e-3)
    return dict(params=m.params, m1=m.m1, m2=m.m2, packs=m.packs)


# arithmetic operations of one walker-step: draws (two Philox4x32-10 blocks are about 250), the
# potential, the branching weight; importance sampling evaluates the trial and its derivatives
# at two points
OPS = {('oscillator', 'plain'): 300, ('water', 'plain'): 400, ('water', 'is'): 900, ('water', 'learned'): 900,
       ('water', 'continuous'): 400, ('cluster', 'plain'): 900, ('cluster', 'is'): 1900}
MLP_OPS = {('water', 128): 66_560, ('water', 256): 264_192, ('cluster', 128): 69_632, ('cluster', 256): 270_336}


def work(case):
    kind = case['kind']
    if kind == 'sim':
        n, np_ = case['n'], 3 if case['system'] == 'oscillator' else 3 * len(MOLECULES[case['system']]['el'])
        ops = OPS[case['system'], case['form']]
        if case['form'] == 'learned':
            ops += MLP_OPS['water', 128]
        return dict(bytes=16 * n * np_ + 16 * case['steps'], flops=ops * n * case['steps'])
    d = 3 if case['system'] == 'water' else 15
    h = case['hidden']
    size = h * d + 2 * h * h + 4 * h + 1
    if kind == 'energy':
        np_ = 9 if case['system'] == 'water' else 18
        return dict(bytes=case['n'] * (np_ * (4 if case['precision'] == 'fp32' else 8) + 8) + 4 * size,
                    flops=case['n'] * MLP_OPS[case['system'], h])
    if kind == 'grads':
        return dict(bytes=4 * (case['n'] * (d + 2) + 2 * size), flops=3 * case['n'] * MLP_OPS[case['system'], h])
    return dict(bytes=4 * 7 * size + 2 * (32 * h + 4 * h * h), flops=12 * size)


def exact(case, seed):
    kind, system = case['kind'], case['system']
    if kind == 'sim':
        return None  # a stochastic trajectory
    if kind == 'adam':
        return _exact_adam(case, seed)
    w = {k: torch.from_numpy(v).cuda().double() for k, v in _weights(system, case['hidden'], seed).items()}
    if kind == 'grads':
        xt, t = _batch(system, case['n'], seed)
        for v in w.values():
            v.requires_grad_(True)
        y = _network(w, xt.t().double())
        loss = ((y - t.double()) ** 2).mean()
        loss.backward()
        g = torch.cat([w[k].grad.reshape(-1) for k in ('W0', 'b0', 'W1', 'b1', 'W2', 'b2', 'w3', 'b3')])
        return dict(loss=loss.detach(), y=y.detach(), grads=g)
    q = _description(system)
    x = torch.from_numpy(_walkers(system, case['n'], seed, 0.08)).cuda()
    if case['precision'] == 'fp32':
        x = x.float().double()
    c = {k: torch.from_numpy(np.asarray(q[k])).cuda().double() for k in ('mean', 'xinv', 'lo', 'hi', 'quad')}
    out = []
    for xs in x.split(100_000):
        f = _features(MOLECULES[system], xs)
        xn = (f - c['mean']) * c['xinv']
        d = xn.shape[1]
        base = c['quad'][0] + xn @ c['quad'][1:1 + d]
        k = 1 + d
        for i in range(d):
            base = base + xn[:, i] * (xn[:, i:] @ c['quad'][k:k + d - i])
            k += d - i
        v = base + q['ymean'] + q['ystd'] * _network(w, xn)
        off = ((f < c['lo']) | (f > c['hi'])).any(1)
        out.append(torch.where(off, _potential(system, xs), v))
    return torch.cat(out)


def _exact_adam(case, seed):
    flat = _weights(case['system'], case['hidden'], seed)
    p = np.concatenate([flat[k].ravel() for k in ('W0', 'b0', 'W1', 'b1', 'W2', 'b2', 'w3', 'b3')]).astype(np.float64)
    g = torch.Generator().manual_seed(seed % (1 << 62))
    gr = (1e-3 * torch.randn(p.size, generator=g)).numpy().astype(np.float64)
    m1 = (1e-3 * torch.randn(p.size, generator=g)).numpy().astype(np.float64)
    m2 = (1e-6 * torch.rand(p.size, generator=g)).numpy().astype(np.float64)
    t = int(case.get('seed_step', 1000)) + 1
    m1 = 0.9 * m1 + 0.1 * gr
    m2 = 0.999 * m2 + 0.001 * gr ** 2
    p = p - 1e-3 * (m1 / (1 - 0.9 ** t)) / (np.sqrt(m2 / (1 - 0.999 ** t)) + 1e-8)
    return dict(params=p, m1=m1, m2=m2, packs=None)
