"""The Vogels, Evans and Custom rules driven by spikes inside the persistent kernel, bit-exact
against the FP32 oracle: rasters, membranes, rings, weights and traces, where the form can go
wrong -- one and several wavefronts of neurons per partition (lists polled by quads or staged),
groups of one step to 32, several spikes of a unit per group, inputs in the rule, every weight
format, weights set out of range (the next group then runs per synapse), groups without
plasticity in between, and the networks that have to stay on the per-synapse form."""
import numpy as np
import pytest

import oracle_py
from spike_amd import abi, builders
from spike_amd.netdesc import Rule, RULE_CUSTOM, RULE_EVANS, RULE_VOGELS, SYN_CONDUCTANCE, SYN_CURRENT, SYN_VOLTAGE, \
    WEIGHTS_BF16, WEIGHTS_FP16, WEIGHTS_FP32
from test_gpu_parity import _compare

pytestmark = pytest.mark.gpu


def _rule(kind, syn, w_max, nearest):
    if kind == RULE_VOGELS:
        return Rule(kind, syn, builders.vogels_params(lr=w_max * 1e-2, rate=20.0))
    if kind == RULE_EVANS:
        return Rule(kind, syn, builders.evans_params())
    return Rule(kind, syn, builders.custom_params(a_star=1e-3, w_max=w_max, learning_rate=w_max * 1e-2, nearest=nearest))


def _net(rule, n=97, n_inputs=41, dmin=3, kind=SYN_VOLTAGE, labels=1, nearest=0, fmt=WEIGHTS_FP32, tref=2e-3, seed=3,
         longer=False):
    if kind == SYN_VOLTAGE:
        cond, w_max = dict(whi=3e-3), 4e-3
    else:
        cond, w_max = dict(wlo=0.0, whi=1.0, scale=4e-9 if kind == SYN_CONDUCTANCE else 2e-12), 1.5
    d = builders.random_net(n_neurons=n, n_inputs=n_inputs, p=0.25, seed=seed, dmin=dmin, dmax=dmin + 5, kind=kind,
                            n_labels=labels, input_rate=400.0, tref=tref, **cond)
    rng = np.random.default_rng(seed + 1)
    syn = rng.permutation(rng.choice(d.n_synapses, size=d.n_synapses // 2, replace=False)).astype(np.int64)
    d.delay[syn] = dmin
    if longer:
        d.delay[syn[7]] = dmin + 1
    d.rules.append(_rule(rule, syn, w_max, nearest))
    d.weight_format = fmt
    return d


def _pieces(d, partitions, by_events):
    gpu = abi.Network(d, partitions=partitions)
    ora = oracle_py.OracleNetwork(d, precision=32)
    assert gpu.info().fused == 1, gpu.fused_status()
    G = d.timestep_grouping()
    long = max(20, 240 // G)
    t = 0.0
    for k, ng in enumerate([long, 1, 7, long // 2]):
        if k == 3:
            w = gpu.weights()
            w[d.rules[0].synapses[::5]] = np.float32(-1e-3)
            w[d.rules[0].synapses[1::5]] = np.float32(1.25)
            gpu.set_weights(w)
            ora.set_weights(w)
        plastic = k != 2
        tm = gpu.run(t, ng, plasticity=plastic)
        # one launch per synapse after prepare and set_weights, then one by spikes
        assert tm.kernel_launches == (2 if by_events and k in (0, 3) else 1)
        ora.run(t, ng, plasticity=plastic)
        t = float(d.group_time(t, ng))
        _compare(gpu, ora, d, f"piece {k}")
    for s in range(10):
        gpu.step_group(d.group_time(t, s))
    ora.run(t, 10)
    t = float(d.group_time(t, 10))
    _compare(gpu, ora, d, "steps")
    gpu.run(t, 5)
    ora.run(t, 5)
    _compare(gpu, ora, d, "after steps")


RULES = [RULE_VOGELS, RULE_EVANS, RULE_CUSTOM]


@pytest.mark.parametrize("partitions", [0, 1, 5, 97])
@pytest.mark.parametrize("rule,nearest,fmt", [(RULE_VOGELS, 0, WEIGHTS_FP32), (RULE_EVANS, 0, WEIGHTS_FP16),
                                              (RULE_CUSTOM, 1, WEIGHTS_BF16), (RULE_CUSTOM, 0, WEIGHTS_FP32)])
def test_partitions(rule, nearest, fmt, partitions):
    _pieces(_net(rule, nearest=nearest, fmt=fmt), partitions, True)


@pytest.mark.parametrize("rule", RULES)
@pytest.mark.parametrize("dmin", [1, 16, 17, 32])
def test_group_lengths(rule, dmin):
    # a refractory time under half a group: several spikes of a neuron per group
    _pieces(_net(rule, dmin=dmin, tref=4e-4, n=150), 0, True)


@pytest.mark.parametrize("rule", RULES)
@pytest.mark.parametrize("kind,labels", [(SYN_CONDUCTANCE, 1), (SYN_CONDUCTANCE, 2), (SYN_CURRENT, 2),
                                         (SYN_CONDUCTANCE, 3)])
def test_synapse_kinds(rule, kind, labels):
    _pieces(_net(rule, kind=kind, labels=labels, dmin=11), 0, True)


@pytest.mark.parametrize("case", ["a longer delay", "a group of 33 steps", "constants that are not finite"])
def test_networks_that_stay_per_synapse(case):
    d = _net(RULE_VOGELS, dmin=33 if "33" in case else 4, longer="longer" in case)
    if "finite" in case:
        d.rules[0].params["targetrate"] = float("inf")
    _pieces(d, 3, False)


def test_times_that_skip_steps():
    """Group times in float32 that round to steps with gaps: the rule runs per synapse (one
    launch, also where the first group is not one that has to)."""
    d = _net(RULE_VOGELS, dmin=2)
    steps = [round(float(d.group_time(1500.0, s) / np.float32(d.dt))) for s in range(30)]
    assert (np.diff(steps) != 2).any()
    gpu = abi.Network(d, partitions=3)
    assert gpu.run(0.0, 20).kernel_launches == 2
    assert gpu.run(1500.0, 30).kernel_launches == 1
    gpu = abi.Network(d, partitions=3)
    assert gpu.run(1500.0, 30).kernel_launches == 1
