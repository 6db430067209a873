"""The weight-dependent rule driven by spikes inside the persistent kernel, bit-exact against
the FP32 oracle: rasters, membranes, rings, weights and traces, where the form can go wrong --
one and several wavefronts of neurons per partition (lists polled by quads or staged), groups
of one and more steps, inputs in the rule or beside it, several labels, every weight format,
weights set below zero (the next group then runs per synapse), and the networks that have to
stay on the per-synapse form."""
import numpy as np
import pytest

import oracle_py
from spike_amd import abi, builders
from spike_amd.netdesc import Rule, RULE_WD, SYN_CONDUCTANCE, SYN_CURRENT, SYN_VOLTAGE, WEIGHTS_BF16, WEIGHTS_FP16, \
    WEIGHTS_FP32
from test_gpu_parity import _compare

pytestmark = pytest.mark.gpu


def _net(n=97, n_inputs=41, dmin=1, dmax=6, kind=SYN_VOLTAGE, labels=1, inputs_in_rule=True, nearest=0,
         fmt=WEIGHTS_FP32, tref=2e-3, seed=3):
    cond = dict(wlo=0.0, whi=1.0, scale=4e-9 if kind == SYN_CONDUCTANCE else 2e-12) if kind != SYN_VOLTAGE else {}
    d = builders.random_net(n_neurons=n, n_inputs=n_inputs, p=0.25, seed=seed, dmin=dmin, dmax=dmax, kind=kind,
                            n_labels=labels, input_rate=400.0, tref=tref, **(cond or dict(whi=3e-3)))
    rng = np.random.default_rng(seed + 1)
    can = np.arange(d.n_synapses) if inputs_in_rule else np.nonzero(d.pre >= 0)[0]
    syn = rng.permutation(rng.choice(can, size=len(can) // 2, replace=False)).astype(np.int64)
    w_max = 4e-3 if kind == SYN_VOLTAGE else 1.5
    d.rules.append(Rule(RULE_WD, syn, builders.wd_params(lam=1e-2, alpha=2.02, w_max=w_max, nearest=nearest)))
    d.weight_format = fmt
    return d


def _pieces(d, partitions, by_events):
    gpu = abi.Network(d, partitions=partitions)
    ora = oracle_py.OracleNetwork(d, precision=32)
    assert gpu.info().fused == 1, gpu.fused_status()
    t = 0.0
    for k, ng in enumerate([120, 1, 60]):
        if k == 2:
            w = gpu.weights()
            w[d.rules[0].synapses[::5]] = np.float32(-1e-3)
            gpu.set_weights(w)
            ora.set_weights(w)
        tm = gpu.run(t, ng)
        # one launch per synapse after prepare and set_weights, then one by spikes
        assert tm.kernel_launches == (2 if by_events and k != 1 else 1)
        ora.run(t, ng)
        t = float(d.group_time(t, ng))
        _compare(gpu, ora, d, f"piece {k}")
    for s in range(30):
        gpu.step_group(d.group_time(t, s))
    ora.run(t, 30)
    _compare(gpu, ora, d, "steps")


@pytest.mark.parametrize("partitions", [0, 1, 5, 97])
@pytest.mark.parametrize("nearest,fmt", [(0, WEIGHTS_FP32), (1, WEIGHTS_FP16), (0, WEIGHTS_BF16)])
def test_groups_of_one_step(partitions, nearest, fmt):
    _pieces(_net(nearest=nearest, fmt=fmt), partitions, True)


@pytest.mark.parametrize("partitions", [0, 2])
@pytest.mark.parametrize("dmin,fmt", [(2, WEIGHTS_FP32), (7, WEIGHTS_FP16)])
def test_groups_of_several_steps(partitions, dmin, fmt):
    _pieces(_net(dmin=dmin, dmax=dmin + 9, inputs_in_rule=False, fmt=fmt, n=150), partitions, True)


@pytest.mark.parametrize("kind,labels", [(SYN_VOLTAGE, 3), (SYN_CONDUCTANCE, 1), (SYN_CONDUCTANCE, 2), (SYN_CURRENT, 2)])
def test_synapse_kinds(kind, labels):
    _pieces(_net(kind=kind, labels=labels), 0, True)


@pytest.mark.parametrize("case", ["inputs in a rule of several steps", "two spikes per group"])
def test_networks_that_stay_per_synapse(case):
    d = _net(dmin=3, dmax=6) if case.startswith("inputs") else _net(dmin=8, dmax=9, inputs_in_rule=False, tref=4e-4)
    _pieces(d, 3, False)


@pytest.mark.parametrize("form", ["persistent", "launches", "steps"])
@pytest.mark.parametrize("dmin", [1, 3])
@pytest.mark.parametrize("start", ["late", "again", "half a step back"])
def test_spikes_that_count_in_two_groups(start, dmin, form):
    """Groups whose float32 start is not clear of the group before: beyond 1024 s, where times no
    longer resolve a step, and runs that begin on the last group's time again or half a step
    before it.  The rule reads a spike's step from its time, so the earlier group's spikes count
    in these groups, too, and their units have to be walked although they did not spike.  The
    persistent kernel keeps its input ring by steps that follow each other and is compared with
    its own per-synapse form (a second rule, which changes nothing, takes the network there)."""
    def net():
        d = _net(dmin=dmin, dmax=dmin + 5, inputs_in_rule=dmin == 1)
        d.monitors = []   # (records of one time in several groups come in the order of the drains)
        return d

    d = net()
    gpu = abi.Network(d, partitions=3)
    if form == "persistent":
        e = net()
        other = np.setdiff1d(np.arange(e.n_synapses), e.rules[0].synapses)[:1]
        e.rules.append(Rule(RULE_WD, other, builders.wd_params(lam=0.0)))
        ref = abi.Network(e, partitions=3)
        assert ref.info().fused == 1
    else:
        ref = oracle_py.OracleNetwork(d, precision=32)

    def both(t, ng):
        ref.run(t, ng)
        if form == "steps":
            for s in range(ng):
                gpu.step_group(d.group_time(t, s))
        else:
            gpu.run(t, ng, force_launches=form == "launches")

    both(0.0, 50)
    last = np.float32(d.group_time(0.0, 49))
    t = {"late": np.float32(1500.0), "again": last, "half a step back": last - np.float32(0.45) * np.float32(d.dt)}[start]
    if start == "late" and dmin == 1:
        assert any(d.group_time(t, s) == d.group_time(t, s + 1) for s in range(60))
    both(float(t), 60)
    _compare(gpu, ref, d, f"{start} {form}")
