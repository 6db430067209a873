"""Groups enqueued one at a time (spk_step_group: two launches a group, monitors recorded where
the spikes are made), bit-exact against the FP32 oracle at the edges of their chunks: groups of
one step, of whole and broken 16-step chunks, of more than 64 steps, more monitors than the
unit kernels record for, rules between the two launches, steps mixed with runs and resets."""
import numpy as np
import pytest

import oracle_py
from spike_amd import abi, builders
from spike_amd.netdesc import Rule, RULE_VOGELS, RULE_WD, SYN_CONDUCTANCE, SYN_VOLTAGE
from test_gpu_parity import _compare

pytestmark = pytest.mark.gpu


def _check(d, ng, plastic=True):
    gpu = abi.Network(d)
    ora = oracle_py.OracleNetwork(d, precision=32)
    for rep in range(2):
        for s in range(ng):
            gpu.step_group(d.group_time(0.0, s), plasticity=plastic)
        t = float(d.group_time(0.0, ng))
        gpu.run(t, 3, plasticity=plastic)
        gpu.step_group(d.group_time(t, 3), plasticity=plastic)
        ora.run(0.0, ng, plastic)
        ora.run(t, 4, plastic)
        _compare(gpu, ora, d, f"pass {rep}")
        gpu.reset_state()
        ora.reset_state()
    return gpu


@pytest.mark.parametrize("dmin,dmax", [(1, 5), (3, 9), (16, 20), (17, 40), (70, 80)])
@pytest.mark.parametrize("kind,labels", [(SYN_VOLTAGE, 1), (SYN_CONDUCTANCE, 2)])
def test_group_lengths(kind, labels, dmin, dmax):
    more = dict(scale=3e-9, whi=1.0) if kind == SYN_CONDUCTANCE else dict(whi=4e-3)
    d = builders.random_net(n_neurons=131, n_inputs=67, p=0.2, seed=dmin, dmin=dmin, dmax=dmax, kind=kind,
                            n_labels=labels, input_rate=300.0, ext_rate=1500.0 if kind == SYN_VOLTAGE else 0.0,
                            ext_w=1e-3, **more)
    _check(d, max(12, 300 // dmin))


def test_more_monitors_than_the_unit_kernels_record_for():
    d = builders.random_net(n_neurons=70, n_inputs=130, seed=5, dmin=2, dmax=6, input_rate=400.0, whi=4e-3,
                            monitors=(0, 0, 1, 0, 0, 0, 1))
    gpu = _check(d, 100)
    assert gpu.info().n_monitors == 7


@pytest.mark.parametrize("rule,dmin", [(RULE_WD, 1), (RULE_WD, 3), (RULE_VOGELS, 4)])
def test_rules(rule, dmin):
    d = builders.random_net(n_neurons=96, n_inputs=48, p=0.25, seed=9, dmin=dmin, dmax=dmin + 4, input_rate=500.0,
                            whi=3e-3)
    syn = np.arange(0, d.n_synapses, 2, dtype=np.int64)
    p = builders.wd_params(w_max=4e-3) if rule == RULE_WD else builders.vogels_params(lr=1e-5)
    d.rules.append(Rule(rule, syn, p))
    _check(d, 120)


@pytest.mark.parametrize("fmt", [0, 1, 2])
@pytest.mark.parametrize("p", [0.0, 0.002, 0.21])
def test_weights_out_and_in(fmt, p):
    """Weights read and set in the caller's (shuffled) order, no synapses included."""
    d = builders.random_net(n_neurons=77, n_inputs=19, p=p, seed=3, whi=1.0, monitors=())
    o = np.random.default_rng(5).permutation(d.n_synapses)
    d.pre, d.post, d.weight, d.delay = d.pre[o], d.post[o], d.weight[o], d.delay[o]
    d.weight_format = fmt
    d.grouping = 1
    gpu = abi.Network(d)
    if fmt:
        d0 = gpu.weights()
        assert np.all(np.abs(d0 - d.weight) <= 0.004 * d.weight + 1e-7)   # half a step of 8 bits
    else:
        assert np.array_equal(gpu.weights(), d.weight)
    w = (np.arange(d.n_synapses) % 128 - 64).astype(np.float32)           # exact in every format
    gpu.set_weights(w)
    assert np.array_equal(gpu.weights(), w)
