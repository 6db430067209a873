"""Order of a drained monitor's records: (time, id), whether the device or the host orders them.
Populations around the 32-unit words, record counts around the smallest that the device orders,
time ranges of one and several tiles, late starts, and the stores that have to be ordered on
the host: records that occur twice, and steps past those whose times name them."""
import numpy as np
import pytest

import oracle_py
from spike_amd import abi, builders

pytestmark = pytest.mark.gpu


def _net(n_inputs, rate, dmin=1, seed=4, **kw):
    return builders.random_net(n_neurons=20, n_inputs=n_inputs, p=0.05, seed=seed, dmin=dmin, dmax=dmin + 3,
                               input_rate=rate, monitors=(1, 0), **kw)


@pytest.mark.parametrize("n_inputs", [1, 31, 32, 33, 700])
@pytest.mark.parametrize("start,groups", [(0.0, 900), (3.25, 900), (0.0, 40)])
def test_raster_equals_oracle(n_inputs, start, groups):
    d = _net(n_inputs, 2000.0 if n_inputs > 1 else 5000.0)
    gpu = abi.Network(d)
    ora = oracle_py.OracleNetwork(d, precision=32)
    for k in range(2):
        t = float(d.group_time(start, k * groups))
        gpu.run(t, groups)
        ora.run(t, groups)
    for m in (0, 1):
        gi, gt = gpu.take_spikes(m)
        oi, ot = ora.take_spikes(m)
        assert np.array_equal(gi, oi) and np.array_equal(gt, ot)
    assert len(gpu.take_spikes(0)[0]) == 0


@pytest.mark.parametrize("extra", [-1, 0, 1])
def test_store_around_the_smallest_device_order(extra):
    """Exactly 2048 + extra records: every input fires at every step but the first."""
    n = 128
    steps = 17    # 16 firing steps x 128 inputs = 2048
    d = _net(n, 1e9)
    d.rates = np.full((1, n), np.float32(1e9), np.float32)
    if extra < 0:
        d.rates[0, 5] = 0.0
    gpu = abi.Network(d)
    ora = oracle_py.OracleNetwork(d, precision=32)
    gpu.run(0.0, steps + (extra > 0))
    ora.run(0.0, steps + (extra > 0))
    gi, gt = gpu.take_spikes(0)
    oi, ot = ora.take_spikes(0)
    assert len(gi) == {-1: 2048 - 16, 0: 2048, 1: 2048 + 128}[extra]
    assert np.array_equal(gi, oi) and np.array_equal(gt, ot)


def test_records_collected_twice_stay_twice():
    d = _net(300, 2000.0)
    gpu = abi.Network(d)
    ora = oracle_py.OracleNetwork(d, precision=32)
    for s in range(60):
        t = d.group_time(0.0, s)
        gpu.step_phases(t)
        abi.check(gpu.lib.spk_collect_spikes(gpu.h, gpu.monitor_ids[0], float(t)))
        ora.step_phases(t)
    gi, gt = gpu.take_spikes(0)
    oi, ot = ora.take_spikes(0)
    assert len(oi) > 2048
    assert np.array_equal(gi, np.repeat(oi, 2)) and np.array_equal(gt, np.repeat(ot, 2))


def test_times_past_the_steps_they_name():
    d = _net(300, 2000.0)
    gpu = abi.Network(d)
    start = 150.0    # step 1 500 000
    gpu.run(start, 100)
    gi, gt = gpu.take_spikes(0)
    assert len(gi) > 2048
    o = np.lexsort((gi, gt))
    assert np.array_equal(o, np.arange(len(gi)))
    ora = oracle_py.OracleNetwork(d, precision=32)
    ora.run(start, 100)
    oi, ot = ora.take_spikes(0)
    assert np.array_equal(gi, oi) and np.array_equal(gt, ot)


@pytest.mark.parametrize("extra", [-1, 0, 1])
def test_store_around_the_line_between_host_and_device(extra):
    """Exactly 6144 + extra records of 192 inputs that fire at every step but the first."""
    n = 192
    steps = 33    # 32 firing steps x 192 inputs = 6144
    d = _net(n, 1e9)
    d.rates = np.full((1, n), np.float32(1e9), np.float32)
    if extra < 0:
        d.rates[0, 5] = 0.0
    gpu = abi.Network(d)
    ora = oracle_py.OracleNetwork(d, precision=32)
    gpu.run(0.0, steps + (extra > 0))
    ora.run(0.0, steps + (extra > 0))
    gi, gt = gpu.take_spikes(0)
    oi, ot = ora.take_spikes(0)
    assert len(gi) == {-1: 6144 - 32, 0: 6144, 1: 6144 + 192}[extra]
    assert np.array_equal(gi, oi) and np.array_equal(gt, ot)
