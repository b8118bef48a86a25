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
