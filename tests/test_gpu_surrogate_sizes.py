"""Sizes at which the surrogate kernels' tilings end: single walkers, one more and one less than a
tile, a wave's and a workgroup's share."""
import numpy as np
import pytest

from oracle import mlp as O
from oracle import pes as P

pytestmark = pytest.mark.gpu

WATER, CLUSTER = ['H', 'H', 'O'], ['O', 'H', 'H', 'O', 'H', 'H']


def walkers(elements, n, seed):
    eq = P.water_eq() if len(elements) == 3 else P.cluster6_eq()
    return eq[None] + np.random.RandomState(seed).normal(0, 0.08, (n,) + eq.shape)


def surface(elements):
    return P.morse_bend if len(elements) == 3 else P.cluster6


def network(m, x):
    """The oracle's network on the model's normalised features of x (float32)."""
    d = m.desc
    f = O.descriptor(x, m.zs, m.sorted_atoms, m.sorted_groups).astype(np.float32)
    mean, inv = (np.array(v[:m.D], np.float32) for v in (d.xmean, d.xinv))
    net = O.MLP(m.D, m.H)
    net.p = {k: v.astype(np.float32) for k, v in m.param_dict().items()}
    return net, ((f - mean) * inv).astype(np.float32)


@pytest.mark.parametrize('elements,hidden', [(WATER, 128), (CLUSTER, 128), (WATER, 256), (CLUSTER, 256)])
@pytest.mark.parametrize('precision', ['fp32', 'fp64'])
def test_energy_sizes(elements, hidden, precision):
    """A large batch against the oracle (2e-3 of the spread: both sides round the same operands to
    bfloat16), then every prefix bit for bit: a walker's energy depends on nothing but itself.
    Walkers outside the range get the analytic potential wherever they lie in a tile."""
    import torch
    import pyvibdmc_amd as pv
    from pyvibdmc_amd import _native as N
    n = 140_003
    x, pes = walkers(elements, n, 3), surface(elements)
    m = pv.SurrogateModel(elements, hidden=hidden, seed=4)
    m.set_normalisation(x[:20000], pes(x[:20000]))
    fp = torch.float32 if precision == 'fp32' else torch.float64
    planes = torch.from_numpy(x).cuda().reshape(n, -1).t().contiguous().to(fp).contiguous()
    fallback = pv.MorseBendTriatomic() if len(elements) == 3 else pv.TwoMonomerCluster()

    def energy(count, use_range):
        m.desc.use_range = use_range
        out = torch.full((count + 8,), float('nan'), dtype=torch.float64, device='cuda')
        m.energy_planes(planes.data_ptr(), n, None, count, out, N.PVD_FP32 if fp == torch.float32 else N.PVD_FP64,
                        fallback)
        v = out.cpu().numpy()
        assert np.isnan(v[count:]).all()
        return v[:count]

    whole = energy(n, 0)
    net, xn = network(m, x[-3000:])
    ref = net.forward(xn)[0] * m.desc.ystd + m.desc.ymean
    assert np.linalg.norm(whole[-3000:] - ref) < 2e-3 * np.linalg.norm(ref - ref.mean())
    sizes = (1, 15, 16, 17, 31, 32, 33, 64, 65, 511, 512, 513, 545, 8191, 8193, 65_537, 131_073)
    for k in sizes:
        np.testing.assert_array_equal(energy(k, 0), whole[:k], err_msg=str(k))
    mixed = energy(n, 1)
    out = mixed != whole
    assert 10 < out.sum() < n // 2
    # an analytic energy of walkers as the device holds them, to its own rounding
    xd = planes.t().double().cpu().numpy().reshape(x.shape)[out]
    np.testing.assert_allclose(mixed[out], pes(xd), rtol=0, atol=1e-6 if precision == 'fp32' else 1e-12)
    for k in sizes:
        np.testing.assert_array_equal(energy(k, 1), mixed[:k], err_msg=str(k))


@pytest.mark.parametrize('features,hidden', [(1, 128), (3, 128), (15, 256), (32, 128), (32, 256), (17, 256)])
@pytest.mark.parametrize('offset', [0, 1])
def test_adam_pack_equals_adam_then_pack(features, hidden, offset):
    """The one-pass update against pvd_mlp_adam and pvd_mlp_pack, bit for bit (the same operations),
    from aligned buffers and from ones at an odd float (which take the two calls)."""
    import ctypes
    import torch
    from pyvibdmc_amd import _native as N
    from pyvibdmc_amd.surrogate import MLPDesc, _lib
    lib = _lib()
    size = int(lib.pvd_mlp_param_count(features, hidden))
    g = torch.Generator().manual_seed(features * hidden)
    base = [torch.randn(size + offset, generator=g), 1e-3 * torch.randn(size + offset, generator=g),
            1e-6 * torch.rand(size + offset, generator=g), 1e-3 * torch.randn(size + offset, generator=g)]
    results = []
    for fused in (False, True):
        p, m1, m2, gr = (b.cuda()[offset:] for b in base)
        packs = torch.full((int(lib.pvd_mlp_pack_bytes(hidden)),), 0x5A, dtype=torch.uint8, device='cuda')
        d = MLPDesc()
        d.D, d.H, d.params, d.packs = features, hidden, p.data_ptr(), packs.data_ptr()
        for t in (1, 2, 1000):
            if fused:
                rc = lib.pvd_mlp_adam_pack(ctypes.byref(d), m1.data_ptr(), m2.data_ptr(), gr.data_ptr(), 1e-3, 0.9, 0.999,
                                           1e-8, t, N.stream_handle())
            else:
                rc = lib.pvd_mlp_adam(p.data_ptr(), m1.data_ptr(), m2.data_ptr(), gr.data_ptr(), size, 1e-3, 0.9, 0.999,
                                      1e-8, t, N.stream_handle()) or lib.pvd_mlp_pack(ctypes.byref(d), N.stream_handle())
            assert rc == 0
        results.append([v.cpu() for v in (p, m1, m2, packs)])
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.parametrize('elements,hidden', [(WATER, 128), (WATER, 256), (CLUSTER, 128), (CLUSTER, 256)])
@pytest.mark.parametrize('n', [1, 2, 31, 33, 255, 257, 511, 513, 4099])
def test_gradient_sizes(elements, hidden, n):
    """Batches at the ends of the tiles (32), slices (256, 512) and loss parts (256) against the
    oracle.  Both sides round the same operands to bfloat16; the accumulation order flips a few of
    those roundings, each of up to 2^-8 of its value: a tensor is held to that, and the mean over a
    large batch to 5e-4.  Nothing is written past the outputs."""
    import ctypes
    import torch
    import pyvibdmc_amd as pv
    from pyvibdmc_amd import _native as N
    from pyvibdmc_amd.surrogate import _lib
    lib = _lib()
    m = pv.SurrogateModel(elements, hidden=hidden, seed=5)
    x, pes = walkers(elements, 5000, 6), surface(elements)
    m.set_normalisation(x, pes(x))
    xt = m.features(x[:n], normalise=True)
    t = torch.from_numpy(((pes(x[:n]) - m.desc.ymean) / m.desc.ystd).astype(np.float32)).cuda()
    parts = (n + 255) // 256
    ws = torch.full((int(lib.pvd_mlp_workspace_bytes(m.D, hidden, n)) + 4096,), 0xA5, dtype=torch.uint8, device='cuda')
    g, y = (torch.full((k + 16,), 7.0, dtype=torch.float32, device='cuda') for k in (m.grads.numel(), n))
    lp, loss = (torch.full((k + 4,), 7.0, dtype=torch.float64, device='cuda') for k in (parts, 1))
    rc = lib.pvd_mlp_loss_grads(ctypes.byref(m.desc), xt.data_ptr(), t.data_ptr(), n, g.data_ptr(), y.data_ptr(),
                                lp.data_ptr(), loss.data_ptr(), ws.data_ptr(), N.stream_handle())
    assert rc == 0, lib.pvd_mlp_last_error()
    assert (g[-16:] == 7).all() and (y[-16:] == 7).all() and (lp[parts:] == 7).all() and (loss[1:] == 7).all()
    assert (ws[-4096:] == 0xA5).all()
    net, xn = network(m, x[:n])
    lo, yo, go = net.loss_grads(xt.cpu().numpy().T.copy(), t.cpu().numpy().astype(np.float64))
    tol = 5e-4 if n > 2000 else 2.0 ** -8
    assert np.linalg.norm(y[:n].cpu().numpy() - yo) <= 2.0 ** -8 * max(np.linalg.norm(yo), np.sqrt(n))
    assert abs(float(loss[0]) - lo) <= 4 * tol * lo
    assert abs(float(lp[:parts].sum()) / n - float(loss[0])) <= 1e-12 * lo
    flat, o, H, D = g.cpu().numpy(), 0, m.H, m.D
    for k, sz in (('W0', H * D), ('b0', H), ('W1', H * H), ('b1', H), ('W2', H * H), ('b2', H), ('w3', H), ('b3', 1)):
        a, b = flat[o:o + sz], go[k].reshape(-1)
        o += sz
        assert np.linalg.norm(a - b) <= 4 * tol * np.linalg.norm(b), k
