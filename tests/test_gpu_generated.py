"""Generated Brunel networks at the edges of the generator's tiles: populations around a tile and
a wavefront, in-degrees that are no multiple of a Philox block, one partition and many, more
sources than the LDS form counts, empty populations -- bit-exact against the oracle's replay of
the rule."""
import numpy as np
import pytest

import oracle_py
from spike_amd import sweep
from sweep_replay import replay_desc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,partitions,eps", [(20, 0, 0.1), (63, 1, 0.1), (65, 3, 0.1), (1250, 4, 0.1), (1999, 0, 0.013),
                                             (2049, 64, 0.1), (33000, 0, 0.0021)])
def test_generated_equals_replay(n, partitions, eps):
    # the product J C_E of the 10^4-neuron network
    p = sweep.SweepPoint(n, 5.0, 2.5, 0.08 / max(1, int(eps * round(0.8 * n))), 12, 77 + n, eps=eps)
    net = sweep.build(p, partitions)
    ora = oracle_py.OracleNetwork(replay_desc(p), precision=32)
    spikes = events = 0
    for k in range(2):
        tm = net.run(float(net.desc.group_time(0.0, 30 * k)), 30, plasticity=False)   # (counts of this run)
        spikes, events = spikes + tm.spikes_neurons, events + tm.external_events
        ora.run(float(net.desc.group_time(0.0, 30 * k)), 30)
    o = ora.counters()
    assert spikes == o["spikes_neurons"] > 0 and events == o["external_events"]
    assert np.array_equal(net.membrane().astype(np.float64), ora.membrane())
    assert np.array_equal(net.ring(), ora.ring())


def _run(p):
    net = sweep.build(p, 0)
    net.stats_begin(10, 600)
    net.run(0.0, 20, plasticity=False)
    v, ring, rate = net.membrane().astype(np.float64), net.ring(), net.stats().rate_hz
    net.close()
    return v, ring, rate


def test_memory_of_closed_networks():
    """Networks that take the memory of closed ones: a little smaller, the same size, another
    in-degree, and from two threads at a time -- each as the oracle's replay."""
    from concurrent.futures import ThreadPoolExecutor
    points = [sweep.SweepPoint(n, 5.0, 2.5, 1e-4, 12, seed, eps=eps)
              for seed, (n, eps) in enumerate([(3000, 0.1), (2900, 0.1), (3000, 0.1), (2950, 0.09), (1500, 0.1)])]
    want = []
    for p in points:
        ora = oracle_py.OracleNetwork(replay_desc(p), precision=32)
        ora.run(0.0, 20)
        want.append((ora.membrane(), ora.ring()))
    one = [_run(p) for p in points]
    with ThreadPoolExecutor(2) as pool:
        two = list(pool.map(_run, points * 2))
    for k, (v, ring, rate) in enumerate(one + two):
        assert np.array_equal(v, want[k % 5][0]) and np.array_equal(ring, want[k % 5][1]), k
        assert rate == one[k % 5][2]
