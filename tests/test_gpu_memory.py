"""What the library does when device memory runs out: calls that found the memory without the
idle memory of closed networks still find it, a refused request leaves no error for a later call
to report, and an object whose buffers could not grow stays usable.  The library refuses requests
itself (spk_refuse_allocations: `pass` requests are served, then `count` refused; a request that is
tried again after the idle memory went back counts twice)."""
import contextlib

import numpy as np
import pytest
import torch

import oracle_py
from spike_amd import abi, builders, mlp, sweep
from spike_amd.netdesc import Rule, RULE_VOGELS
from sweep_replay import replay_desc

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def _refused(count, after=0):
    lib = abi.load()
    lib.spk_refuse_allocations(after, count)
    try:
        yield
    finally:
        lib.spk_refuse_allocations(0, 0)


def _generated(n, seed):
    return sweep.SweepPoint(n, 5.0, 2.5, 1e-4, 12, seed)


def _equals_replay(p, net):
    ora = oracle_py.OracleNetwork(replay_desc(p), precision=32)
    net.run(0.0, 20, plasticity=False)
    ora.run(0.0, 20)
    assert np.array_equal(net.membrane().astype(np.float64), ora.membrane())
    assert np.array_equal(net.ring(), ora.ring())


def test_request_that_succeeds_after_idle_memory_went_back():
    sweep.build(_generated(3000, 1), 0).close()      # leaves idle memory
    p = _generated(7001, 2)
    with _refused(1):
        net = sweep.build(p, 0)
    _equals_replay(p, net)


def test_refused_request_leaves_no_error_behind():
    d = builders.random_net(seed=2, input_rate=400.0, whi=4e-3)
    with _refused(2):
        with pytest.raises(abi.SpikeError, match="error 4"):
            abi.Network(d)
    gpu = abi.Network(d)
    ora = oracle_py.OracleNetwork(d, precision=32)
    gpu.run(0.0, 20)
    ora.run(0.0, 20)
    assert np.array_equal(gpu.membrane().astype(np.float64), ora.membrane())


def test_surrogate_takes_what_idle_memory_gives_back():
    p = mlp.init_params(5, 2)
    x = np.random.default_rng(6).uniform(-1.0, 1.0, (300, mlp.INPUTS)).astype(np.float32)
    ref = mlp.Mlp(2, 256)
    ref.set_params(p)
    want = ref.predict(x)
    with _refused(2):
        with pytest.raises(abi.SpikeError, match="error 4"):
            mlp.Mlp(2, 256)
    sweep.build(_generated(3000, 1), 0).close()
    with _refused(1):
        net = mlp.Mlp(2, 256)
    net.set_params(p)
    assert np.array_equal(net.predict(x), want)


def test_parameters_without_memory_for_a_copy():
    p = mlp.init_params(7, 3)
    bad = p.copy()
    bad[1, 17] = np.nan
    bad[2, 5] = np.inf
    x = np.random.default_rng(8).uniform(-1.0, 1.0, (40, mlp.INPUTS)).astype(np.float32)
    net = mlp.Mlp(3, 128)
    with _refused(100):
        net.set_params(p)
        with pytest.raises(abi.SpikeError, match=f"non-finite parameter at {mlp.PARAMS + 17}$"):
            net.set_params(bad)
    y = net.predict(x)
    assert np.array_equal(net.params(), p)
    net.set_params(p)
    assert np.array_equal(net.predict(x), y)


@pytest.mark.parametrize("served", [0, 1])
def test_surrogate_buffers_that_could_not_grow(served):
    """Rows and results of a prediction, and a training set, after a larger one was refused: the
    sizes that were there before are not taken for memory that is."""
    rng = np.random.default_rng(9)
    x = rng.uniform(-1.0, 1.0, (5000, mlp.INPUTS)).astype(np.float32)
    t = rng.standard_normal((5000, mlp.OUTPUTS)).astype(np.float32)
    net = mlp.Mlp(2, 128)
    net.set_params(mlp.init_params(9, 2))
    y = net.predict(x[:300])
    net.set_data(x[:256], t[:256])
    loss, grads = net.gradients(128)
    with _refused(2, served):
        with pytest.raises(abi.SpikeError, match="error 4"):
            net.predict(x)
    with _refused(2, served):
        with pytest.raises(abi.SpikeError, match="error 4"):
            net.set_data(x, t)
    assert np.array_equal(net.predict(x[:300]), y)
    with pytest.raises(abi.SpikeError, match="training set"):
        net.gradients(128)
    net.set_data(x[:256], t[:256])
    loss1, grads1 = net.gradients(128)
    assert np.array_equal(loss1, loss) and np.array_equal(grads1, grads)


def test_refused_statistics_are_not_asked_for_twice():
    n = 400_000                                  # 28 bytes a neuron: 11 MB
    gpu = abi.Network(builders.large_plastic(n=n, out_degree=2, input_out_degree=2, generated=True))
    with _refused(100):                          # (idle memory of this size may serve it)
        with contextlib.suppress(abi.SpikeError):
            gpu.stats_begin(1, 10)
    free = torch.cuda.mem_get_info()[0]
    gpu.stats_begin(1, 10)
    assert free - torch.cuda.mem_get_info()[0] <= 28 * n + (6 << 20)
    gpu.run(0.0, 10)
    assert gpu.stats().steps == 10


def test_statistics_window_that_could_not_grow():
    d = builders.random_net(seed=2, input_rate=400.0, whi=4e-3, dmin=2, dmax=6)
    gpu, ref = abi.Network(d), abi.Network(d)
    gpu.stats_begin(10, 200)
    gpu.run(0.0, 50)
    assert gpu.stats().spikes > 0
    with _refused(2):
        with pytest.raises(abi.SpikeError, match="error 4"):
            gpu.stats_begin(1, 100_000)
    with pytest.raises(abi.SpikeError, match="never started"):
        gpu.stats()
    t = float(d.group_time(0.0, 50))
    gpu.run(t, 50)                               # no window
    ref.run(0.0, 50)
    ref.run(t, 50)
    t = float(d.group_time(0.0, 100))
    for net in (gpu, ref):
        net.stats_begin(10, 200)
        net.run(t, 60)
    a, b = gpu.stats(), ref.stats()
    assert (a.spikes, a.isi_cv, a.synchrony, a.steps) == (b.spikes, b.isi_cv, b.synchrony, b.steps)


def _monitored():
    d = builders.random_net(n_neurons=700, n_inputs=900, p=0.02, seed=11, input_rate=300.0, whi=4e-3, monitors=(0, 1))
    return d, abi.Network(d), oracle_py.OracleNetwork(d, precision=32)


def _same_rasters(gpu, ora):
    for m in (0, 1):
        for a, b in zip(gpu.take_spikes(m), ora.take_spikes(m)):
            assert len(a) > 0 and np.array_equal(a, b)


def test_monitor_stores_smaller_than_a_whole_run():
    d, gpu, ora = _monitored()
    assert d.timestep_grouping() == 1
    with _refused(2):                            # the store of the first monitor for 1000 groups
        tm = gpu.run(0.0, 600)
    assert tm.kernel_launches == 3               # 256 groups at a time
    ora.run(0.0, 600)
    _same_rasters(gpu, ora)


@pytest.mark.parametrize("refused", [4, 100])
def test_monitor_store_that_could_not_grow(refused):
    """The store of before stays (or, where even that is not to be had, none), and the records of
    the next groups go nowhere else."""
    d, gpu, ora = _monitored()
    with _refused(refused):
        with pytest.raises(abi.SpikeError, match="error 4"):
            gpu.run(0.0, 600)
    gpu.reset_state()
    for s in range(40):
        gpu.step_group(d.group_time(0.0, s))
    ora.run(0.0, 40)
    if refused == 4:
        _same_rasters(gpu, ora)
    else:
        with pytest.raises(abi.SpikeError, match="error 5"):
            gpu.take_spikes(0)
        gpu.lib.spk_monitor_reset(gpu.h, gpu.monitor_ids[0])
        ora.take_spikes(0)
        ora.take_spikes(1)
    gpu.take_spikes(1)
    t = float(d.group_time(0.0, 40))
    gpu.run(t, 100)
    ora.run(t, 100)
    _same_rasters(gpu, ora)


@pytest.mark.parametrize("served", [0, 1, 2, 3, 4, 5, 6])
def test_raster_without_memory_to_order_it_on_the_device(served):
    d, gpu, ora = _monitored()

    def steps(t):
        for s in range(300):
            gpu.step_group(d.group_time(t, s))
        ora.run(t, 300)

    steps(0.0)
    with _refused(100, served):
        _same_rasters(gpu, ora)
    steps(float(d.group_time(0.0, 300)))
    _same_rasters(gpu, ora)


def _weights_name_synapses(gpu, S, fmt):
    """Weights that name their synapse (in two passes of 256 values, exact in every format), set
    and read, whole and every piece's first and last."""
    k = np.arange(S)
    for part in (k % 256, k // 256 % 256, k // 65536):
        w = part.astype(np.float32)
        gpu.set_weights(w)
        assert np.array_equal(gpu.weights(), w), fmt


# (requests refused, after how many served): positions for all synapses first, then the piece,
# each tried twice; a refused piece is tried at a quarter of its size
@pytest.mark.parametrize("refused,served", [(0, 0), (2, 0), (4, 0), (4, 1), (6, 0), (6, 1), (2, 2)])
@pytest.mark.parametrize("fmt", [0, 1, 2])
def test_weights_in_pieces(fmt, refused, served):
    """Weights of a listed network (synapses in shuffled order) with pieces of S, S / 4 and S / 16
    synapses (rounded up: the last one ragged), positions kept or travelling with the piece."""
    d = builders.random_net(n_neurons=331, n_inputs=77, p=0.53, seed=3, whi=1.0, monitors=())
    o = np.random.default_rng(5).permutation(d.n_synapses)
    d.pre, d.post, d.weight, d.delay = d.pre[o], d.post[o], d.weight[o], d.delay[o]
    d.weight_format = fmt
    d.grouping = 1
    assert d.n_synapses > 16 * 4096
    gpu = abi.Network(d)
    with _refused(refused, served):
        w = gpu.weights()
    assert np.array_equal(w, d.weight) if fmt == 0 else np.abs(w - d.weight).max() <= 0.004
    _weights_name_synapses(gpu, d.n_synapses, fmt)


@pytest.mark.parametrize("refused", [0, 2, 4])
@pytest.mark.parametrize("fmt", [0, 1])
def test_weights_of_generated_synapses_in_pieces(fmt, refused):
    d = builders.large_plastic(n=3000, out_degree=30, input_out_degree=31, generated=True)
    d.weight_format = fmt
    gpu, ref = abi.Network(d), abi.Network(d)
    with _refused(refused):
        w = gpu.weights()
    assert np.array_equal(w, ref.weights())
    _weights_name_synapses(gpu, d.n_synapses, fmt)


def test_weights_without_memory_for_any_piece():
    d = builders.random_net(n_neurons=200, n_inputs=80, p=0.7, seed=2)
    assert d.n_synapses > 20480
    gpu = abi.Network(d)
    with _refused(1000):
        with pytest.raises(abi.SpikeError, match="error 4"):
            gpu.weights()
    assert np.array_equal(gpu.weights(), d.weight)


def test_delayed_rule_keeps_what_its_kernels_read():
    """Beside what the per-synapse form has, a Vogels rule that runs by spikes keeps the synapses
    of each target (8 bytes each), a bit per synapse and arrays of a few bytes per unit."""
    n = 2000
    syn = np.arange(n * n, dtype=np.int64)

    def memory(delay_of_one):
        d = builders.random_net(n_neurons=n, n_inputs=0, p=1.0, seed=1, dmin=4, dmax=4, monitors=())
        assert d.n_synapses == n * n
        d.delay[7] = delay_of_one
        d.rules.append(Rule(RULE_VOGELS, syn, builders.vogels_params(lr=1e-5)))
        free = torch.cuda.mem_get_info()[0]
        gpu = abi.Network(d)
        assert gpu.info().fused == 1
        used = free - torch.cuda.mem_get_info()[0]
        gpu.close()
        return used

    memory(4)
    by_spikes, per_synapse = memory(4), memory(5)
    assert 8 * n * n <= by_spikes - per_synapse <= 8 * n * n + n * n // 8 + (6 << 20)


@pytest.mark.parametrize("fmt", [0, 2])
def test_delayed_rule_without_memory_for_its_spike_driven_form(fmt):
    """Whichever request is refused: a network with a delayed rule that can run by spikes is
    refused for as many as one whose rule cannot (it runs per synapse where its lists are not to
    be had), and runs as the oracle does when it is not refused."""
    def net(delay_of_one):
        d = builders.random_net(n_neurons=60, n_inputs=20, p=0.2, seed=4, dmin=3, dmax=3, input_rate=500.0, whi=3e-3)
        d.delay[7] = delay_of_one
        d.rules.append(Rule(RULE_VOGELS, np.arange(d.n_synapses, dtype=np.int64), builders.vogels_params(lr=1e-5)))
        d.weight_format = fmt
        return d

    def outcomes(d):
        ora = oracle_py.OracleNetwork(d, precision=32)
        ora.run(0.0, 30)
        needed = forms = 0
        for served in range(80):
            with _refused(2, served):
                try:
                    gpu = abi.Network(d)
                except abi.SpikeError as e:
                    assert "error 4" in str(e)
                    needed += 1
                    continue
            forms |= gpu.run(0.0, 30).kernel_launches
            assert np.array_equal(gpu.weights().astype(np.float64), ora.weights())
            assert np.array_equal(gpu.membrane().astype(np.float64), ora.membrane())
        return needed, forms

    by_spikes, per_synapse = outcomes(net(3)), outcomes(net(4))
    assert by_spikes[0] == per_synapse[0] > 20
    assert (by_spikes[1], per_synapse[1]) == (3, 1)   # launches of one run: per synapse 1, by spikes 2


def test_memory_of_closed_networks_goes_back_on_request():
    p = _generated(12000, 5)                     # 1200 synapses of 2 bytes a neuron: 29 MB
    abi.release_memory()
    sweep.build(p, 0).close()
    kept = torch.cuda.mem_get_info()[0]
    abi.release_memory()
    assert torch.cuda.mem_get_info()[0] - kept >= 12000 * 1200 * 2
    abi.release_memory()                         # nothing left
    _equals_replay(_generated(1300, 6), sweep.build(_generated(1300, 6), 0))


@pytest.mark.parametrize("fmt", [0, 1, 2])
@pytest.mark.parametrize("synapses", [1, 20479, 20480, 20481])
def test_weights_around_the_line_between_host_and_device(synapses, fmt):
    d = builders.random_net(n_neurons=200, n_inputs=80, p=0.7, seed=3, whi=1.0, monitors=())
    o = np.random.default_rng(5).permutation(d.n_synapses)[:synapses]
    d.pre, d.post, d.weight, d.delay = d.pre[o], d.post[o], d.weight[o], d.delay[o]
    d.weight_format = fmt
    d.grouping = 1
    gpu = abi.Network(d)
    with _refused(1000 if synapses <= 20480 else 0):
        w = gpu.weights()
    assert np.array_equal(w, d.weight) if fmt == 0 else np.abs(w - d.weight).max() <= 0.004
    _weights_name_synapses(gpu, synapses, fmt)
