"""What launching the resident discrete steps costs: the first of a process, and two simulations on
two streams."""
import os
import subprocess
import sys
import threading
import time

import pytest

from tests.conftest import ROOT
from tests.test_gpu_resident import make

pytestmark = pytest.mark.gpu

FIRST = """
import sys, time
sys.path.insert(0, {root!r})
import torch
from tests.test_gpu_resident import make
from pyvibdmc_amd import _native as N
sim = make('water', 5000, 1000, 'fp32')
sim._start()
N.check(N.load().pvd_sim_run(sim._h, 5, N.stream_handle()))
for _ in range(5):
    torch.cuda.synchronize()
    t = time.perf_counter()
    N.check(N.load().pvd_sim_run(sim._h, 150, N.stream_handle()))
    torch.cuda.synchronize()
    print((time.perf_counter() - t) * 1e6)
"""


def test_first_resident_launch_of_a_process():
    """150 steps of 5 000 walkers take 0.7 ms.  The first launch of a process also brings the code to
    the device (0.4 ms a code object and 1 ms a megabyte); a queue of its own would be 3.7 ms more."""
    out = subprocess.run([sys.executable, '-c', FIRST.format(root=ROOT)], capture_output=True, text=True, timeout=100,
                         env=dict(os.environ), cwd=ROOT)
    assert out.returncode == 0, out.stderr
    us = [float(x) for x in out.stdout.split()]
    print('us', us)
    assert us[0] - min(us[1:]) < 3000


def test_small_simulations_on_two_streams_overlap():
    """Two simulations of 5 000 walkers (20 workgroups each) on two streams run beside each other.  Of
    several pairs of streams, as two streams may share one of the four hardware queues, where work is
    done in order."""
    import torch
    from pyvibdmc_amd import _native as N
    lib = N.load()
    sims = [make('water', 5000, 10 ** 6, 'fp32', seed=s) for s in (1, 2)]
    streams = [torch.cuda.Stream() for _ in range(4)]

    def go(i, stream):
        with torch.cuda.stream(stream):
            if not sims[i]._started:
                sims[i]._start()
            N.check(lib.pvd_sim_run(sims[i]._h, 3000, N.stream_handle()))
            stream.synchronize()

    def together(a, b):
        th = [threading.Thread(target=go, args=(i, s)) for i, s in ((0, a), (1, b))]
        [t.start() for t in th]
        [t.join() for t in th]

    def ms(f):
        torch.cuda.synchronize()
        t = time.perf_counter()
        f()
        return (time.perf_counter() - t) * 1e3

    go(0, streams[0]), go(1, streams[0])
    turn = min(ms(lambda: (go(0, streams[0]), go(1, streams[0]))) for _ in range(3))
    both = [ms(lambda: together(a, b)) for k, a in enumerate(streams) for b in streams[k + 1:]]
    print('in turn', turn, 'together', both)
    assert min(both) < 0.8 * turn
    for s in sims:
        assert s._status()[0] == 0


@pytest.mark.parametrize('n', [200_000, 1_000_000])
def test_large_simulations_on_several_streams_take_turns(n):
    """Three simulations whose launches take all CUs each: none waits for another's CUs at its gate, so
    no launch is given up and together they take no longer than in turn."""
    import torch
    from pyvibdmc_amd import _native as N
    from tests.test_gpu_resident_rest import counts
    lib = N.load()
    sims = [make('water', n, 10 ** 6, 'fp32', seed=s) for s in (1, 2, 3)]
    streams = [torch.cuda.Stream() for _ in sims]

    def go(i, steps=1000):
        with torch.cuda.stream(streams[i]):
            if not sims[i]._started:
                sims[i]._start()
            for _ in range(2):
                N.check(lib.pvd_sim_run(sims[i]._h, steps // 2, N.stream_handle()))
            streams[i].synchronize()

    def together():
        th = [threading.Thread(target=go, args=(i,)) for i in range(3)]
        [t.start() for t in th]
        [t.join() for t in th]

    def ms(f):
        torch.cuda.synchronize()
        t = time.perf_counter()
        f()
        return (time.perf_counter() - t) * 1e3

    [go(i, 200) for i in range(3)]
    turn, both = ms(lambda: [go(i) for i in range(3)]), [ms(together) for _ in range(3)]
    print('in turn', turn, 'together', both)
    for s in sims:
        assert s._status()[0] == 0 and counts(s)[1] == 0
    assert min(both) < 1.3 * turn


def test_other_streams_get_their_turn():
    """A million walkers fill the LDS of every CU; a kernel of another stream that needs LDS waits for
    one launch (2 ms), not for all of the 4 000 steps (62 ms).  Of several streams, as one may share a
    hardware queue with the simulation's."""
    import torch
    from pyvibdmc_amd import _native as N
    sim = make('water', 1_000_000, 10 ** 5, 'fp32')
    sim._start()
    a, m = torch.cuda.Stream(), torch.randn(1024, 1024, device='cuda')
    waits = []
    for _ in range(4):
        b = torch.cuda.Stream()
        for timed in (False, True):
            torch.cuda.synchronize()
            if timed:
                N.check(N.load().pvd_sim_run(sim._h, 4000, a.cuda_stream))
                time.sleep(5e-3)
            t = time.perf_counter()
            with torch.cuda.stream(b):
                m @ m
                b.synchronize()
        waits.append((time.perf_counter() - t) * 1e3)
    torch.cuda.synchronize()
    print('ms', waits)
    assert sim._status()[0] == 0
    assert min(waits) < 25


def test_threads_with_plans_of_different_sizes():
    """Two threads on one kernel whose plans ask for different amounts of LDS (with and without the
    descendant tracker): every call is served, and the results are those of the runs alone."""
    import numpy as np
    import torch
    from pyvibdmc_amd import _native as N
    lib = N.load()

    def run(window, stream):
        with torch.cuda.stream(stream):
            sim, st = make('water', 300_000, 10 ** 4, 'fp32', seed=7), N.stream_handle()
            sim._start()
            if window:
                N.check(lib.pvd_sim_desc_begin(sim._h, st))
            for _ in range(60):
                N.check(lib.pvd_sim_run(sim._h, 24, st))
            assert sim._status()[0] == 0
            return sim._get_walkers()[0]

    alone = run(False, torch.cuda.Stream())
    got, streams = [None, None], [torch.cuda.Stream(), torch.cuda.Stream()]

    def work(i):
        got[i] = run(bool(i), streams[i])

    th = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    [t.start() for t in th]
    [t.join() for t in th]
    for g in got:  # the tracker does not change the walkers
        np.testing.assert_array_equal(g, alone)
