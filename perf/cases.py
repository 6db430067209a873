"""Performance cases: what a user of the backend has it do, through the public entry points of
spike_amd.abi, spike_amd.sweep and spike_amd.mlp, from the smallest calls to the largest.

Every simulation case is one trial: the network that prepare() built goes back to its
initial state, runs, and hands back what the program reads (raster, statistics, membranes,
weights).  Weights are kept from trial to trial where the network learns, as in a program
that trains over trials.  Sizes are those of the networks in spike_amd.builders, of the sweep
distribution in spike_amd.sweep and of the surrogate's training and screening calls.
"""
import math

import numpy as np
import torch

from spike_amd import abi, builders, mlp, sweep
from spike_amd.netdesc import WEIGHTS_BF16, WEIGHTS_FP16, WEIGHTS_FP32


def listed():
    return [
        # A front-end program's loop: one spk_step_group call per timestep group, the raster
        # read every 50 groups (the front-end's monitor polling), on a small Brunel network.
        dict(name="front_end_groups", kind="groups", n=2500, groups=100, delay=15),
        # The smallest benchmark network (1000 Poisson inputs -> 1000 conductance LIF, delays
        # from one step, so one exchange per step): latency.
        dict(name="plain_small", kind="plain", groups=1000),
        # Conductance network with two labels and inhibitory plasticity (Vogels-Abbott, 4000
        # neurons), raster and weights read after the trial.
        dict(name="coba_vogels", kind="coba", n=4000, groups=250, weights="fp32"),
        # The flagship: Brunel 10 000 neurons, 1e7 synapses, one simulated second, statistics.
        dict(name="brunel10k", kind="brunel", n=10000, delay=15, groups=666),
        # The example program's encoding of the Brunel network: 10^4 shared Poisson inputs, an
        # odd size, raster read after the trial.
        dict(name="brunel_inputs", kind="inputs", n=5003, delay=15, groups=200),
        # A mid-sized network from the caller's synapse arrays with weight-dependent STDP on
        # E->E, delays 1..20 (one group per step), weights read after the trial.
        dict(name="wd_stdp", kind="stdp", n=6000, out_degree=500, groups=400, weights="fp32"),
        # The largest network: 5e5 neurons, 5.25e8 synapses generated on the device, 16-bit
        # weights, weight-dependent STDP on 3.2e8 of them.
        dict(name="large_plastic", kind="large", n=500000, out_degree=1000, groups=600, weights="fp16"),
        # Another realisation of the external drive for a kept batch of uneven networks.
        dict(name="sweep_realisation", kind="realise", points=64, seconds=0.1),
        # Sweep points from scratch: networks generated, run as one batch, statistics read
        # (the call that makes the surrogate's training data).
        dict(name="sweep_points", kind="points", points=48, seconds=0.1),
        # Screening a few candidate points with the surrogate: latency of a small inference.
        dict(name="predict_small", kind="predict", members=8, rows=100),
        # Screening a large grid: 8 members x 2^18 rows (odd count).
        dict(name="predict_large", kind="predict", members=8, rows=262147),
        # Fitting the surrogate: gradients of the whole ensemble, then optimiser steps at the
        # end of the learning-rate schedule, weights read back.
        dict(name="train", kind="train", members=8, batch=4096, steps=32, data=50000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["groups", "plain", "coba", "brunel", "inputs", "stdp", "large", "realise", "points",
                       "predict", "predict", "train"])
    if kind == "groups":
        return dict(kind=kind, n=_log_int(rng, 500, 2500), groups=rng.randint(50, 100), delay=rng.randint(10, 20))
    if kind == "plain":
        return dict(kind=kind, groups=rng.randint(300, 1000))
    if kind == "coba":
        return dict(kind=kind, n=_log_int(rng, 500, 4000), groups=rng.randint(100, 250),
                    weights=rng.choice(["fp32", "fp32", "fp16", "bf16"]))
    if kind == "brunel":
        return dict(kind=kind, n=_log_int(rng, 1250, 10000), delay=rng.randint(10, 20), groups=rng.randint(300, 666))
    if kind == "inputs":
        return dict(kind=kind, n=_log_int(rng, 1250, 5003), delay=rng.randint(10, 20), groups=rng.randint(100, 200))
    if kind == "stdp":
        return dict(kind=kind, n=_log_int(rng, 1000, 6000), out_degree=_log_int(rng, 100, 500),
                    groups=rng.randint(200, 400), weights=rng.choice(["fp32", "fp16", "bf16"]))
    if kind == "large":
        return dict(kind=kind, n=_log_int(rng, 20000, 500000), out_degree=_log_int(rng, 200, 1000),
                    groups=rng.randint(300, 600), weights=rng.choice(["fp32", "fp16", "bf16"]))
    if kind == "realise":
        return dict(kind=kind, points=_log_int(rng, 4, 64), seconds=round(rng.uniform(0.05, 0.1), 3))
    if kind == "points":
        return dict(kind=kind, points=_log_int(rng, 4, 48), seconds=round(rng.uniform(0.05, 0.1), 3))
    if kind == "predict":
        return dict(kind=kind, members=rng.randint(1, 8), rows=_log_int(rng, 1, 262147))
    return dict(kind=kind, members=rng.randint(1, 8), batch=128 * _log_int(rng, 1, 32), steps=rng.randint(8, 32),
                data=_log_int(rng, 4096, 50000))


_FORMAT = {"fp32": WEIGHTS_FP32, "fp16": WEIGHTS_FP16, "bf16": WEIGHTS_BF16}


def _describe(case, seed):
    """The network description of a single-network case."""
    kind = case["kind"]
    if kind == "plain":
        d = builders.plain_small(seed=seed, monitors=(0, 1))
    elif kind == "coba":
        ne = int(round(0.8 * case["n"]))
        # the in-degree of the 4000-neuron network (p = 0.02) at every size
        d = builders.coba_vogels(n_exc=ne, n_inh=case["n"] - ne, p=min(1.0, 80.0 / case["n"]), seed=seed)
        d.weight_format = _FORMAT[case["weights"]]
    elif kind in ("groups", "brunel", "inputs"):
        ne = int(round(0.8 * case["n"]))
        # in-degree 1000 per neuron of a 10^4-neuron network; smaller networks keep the rule
        # C = eps N and the product J C
        d = builders.brunel(n_exc=ne, n_inh=case["n"] - ne, J=0.1e-3 * 10000 / case["n"], seed=seed,
                            delay_steps=case["delay"], form="reference" if kind == "inputs" else "config",
                            reference_input_rate=20.0 * (case["n"] / 10000 if kind == "inputs" else 1.0),
                            monitors=() if kind == "brunel" else (0,))
    elif kind == "stdp":
        k = case["out_degree"]
        d = builders.large_plastic(n=case["n"], out_degree=k, input_out_degree=k, J=0.1e-3 * 1000 / k,
                                   J_in=2e-3, input_rate=10.0 * 1000 / k, seed=seed, generated=False)
        d.weight_format = _FORMAT[case["weights"]]
    else:
        k = case["out_degree"]
        d = builders.large_plastic(n=case["n"], out_degree=k, input_out_degree=k, J=0.1e-3 * 1000 / k,
                                   J_in=2e-3, input_rate=10.0 * 1000 / k, seed=seed, generated=True)
        d.weight_format = _FORMAT[case["weights"]]
    return d


def _train_inputs(case, seed):
    rng = np.random.default_rng(seed)
    x = rng.uniform(-1.0, 1.0, (case["data"], mlp.INPUTS)).astype(np.float32)
    # smooth targets with noise, standardised, as the surrogate's are
    t = np.stack([np.sin(2.0 * x[:, 0]) + x[:, 1] * x[:, 2], np.cos(x[:, 3]) * x[:, 4], x[:, 0] * x[:, 4]], 1)
    t = (t - t.mean(0)) / t.std(0) + 0.02 * rng.standard_normal(t.shape)
    return x, t.astype(np.float32), mlp.init_params(seed + 1, case["members"])


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("realise", "points"):
        pts = sweep.sample_points(case["points"], seed=1000 + seed)
        state = dict(case=case, seed=seed, points=pts, plan=sweep.default_plan(pts), passes=0)
        if kind == "realise":
            order = state["plan"]["order"]
            nets = [sweep.build(p, P) for p, P in zip(pts, state["plan"]["partitions"])]
            state.update(nets=nets, batch=abi.Batch([nets[k] for k in order]),
                         groups=[pts[k].groups(case["seconds"]) for k in order])
        return state
    if kind == "predict":
        net = mlp.Mlp(case["members"], 1024)
        net.set_params(mlp.init_params(seed + 1, case["members"]))
        x = np.random.default_rng(seed).uniform(-1.0, 1.0, (case["rows"], mlp.INPUTS)).astype(np.float32)
        return dict(case=case, net=net, x=x)
    if kind == "train":
        x, t, p0 = _train_inputs(case, seed)
        net = mlp.Mlp(case["members"], case["batch"])
        net.set_data(x, t)
        return dict(case=case, seed=seed, net=net, p0=p0)
    d = _describe(case, seed)
    return dict(case=case, net=abi.Network(d), desc=d)


# the train case's schedule: the end of the surrogate's cosine schedule (lr_min = 1e-5)
_LR = 1e-5


def _raster(ids, times, units):
    """A raster as the fixed-size arrays (32 records per unit, -1 beyond the last) that a program
    keeps over trials."""
    out = np.full(32 * units, -1, np.int32), np.full(32 * units, -1.0, np.float32)
    out[0][:len(ids)] = ids
    out[1][:len(ids)] = times
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "predict":
        return state["net"].predict(state["x"])
    if kind == "train":
        net = state["net"]
        net.set_params(state["p0"])
        loss, grads = net.gradients(min(case["batch"], (case["data"] // mlp.ROW_TILE) * mlp.ROW_TILE))
        net.train(case["steps"], case["batch"], _LR, _LR, case["steps"], mode=mlp.BATCH_SAMPLED,
                  seed=state["seed"], use_graph=True, record_loss=False)
        return dict(loss=loss, grads=grads, params=net.params())
    if kind == "points":
        r = sweep.run_batched(state["points"], case["seconds"], state["plan"])
        return dict(rate=r.rate, cv=r.cv, sync=r.sync)
    if kind == "realise":
        pts, nets = state["points"], state["nets"]
        state["passes"] += 1
        for p, n in zip(pts, nets):
            abi.check(n.lib.spk_set_seed(n.h, sweep.drive_seed(p, 1 + state["passes"] % 16)))
            n.reset_state()
            n.stats_begin(10, p.groups(case["seconds"]) * p.delay_steps)
        state["batch"].run(np.zeros(len(pts)), state["groups"])
        stats = [n.stats() for n in nets]
        return dict(rate=np.array([s.rate_hz for s in stats]), cv=np.array([s.isi_cv for s in stats]),
                    sync=np.array([s.synchrony for s in stats]),
                    spikes=np.array([s.spikes for s in stats], dtype=np.int64))
    net, d = state["net"], state["desc"]
    net.reset_state()
    if kind == "groups":
        raster = []
        for s in range(case["groups"]):
            net.step_group(d.group_time(0.0, s))
            if s % 50 == 49:
                raster.append(net.drain_spikes(0, cap=60 * d.n_neurons))
        raster.append(net.drain_spikes(0, cap=60 * d.n_neurons))
        ids, times = _raster(*(np.concatenate(x) for x in zip(*raster)), d.n_neurons)
        return dict(ids=ids, times=times, v=net.membrane())
    if kind == "brunel":
        net.stats_begin(10, case["groups"] * d.timestep_grouping())
        t = net.run(0.0, case["groups"], plasticity=False)
        s = net.stats()
        return dict(v=net.membrane(), last=net.last_spike(0), rate=s.rate_hz, cv=s.isi_cv, sync=s.synchrony,
                    counts=np.array([s.spikes, t.synaptic_events, t.external_events], dtype=np.int64))
    t = net.run(0.0, case["groups"])
    out = dict(v=net.membrane(), last=net.last_spike(0),
               counts=np.array([t.spikes_neurons, t.spikes_inputs, t.synaptic_events], dtype=np.int64))
    if kind == "large":
        return out   # 5e8 weights are read once per experiment, not once per trial
    if kind in ("plain", "coba", "inputs"):
        out["ids"], out["times"] = _raster(*net.take_spikes(0), d.n_neurons)
    if kind == "plain":
        out["in_ids"], out["in_times"] = _raster(*net.take_spikes(1), d.n_inputs)
        out["g"] = net.conductances()
    if kind == "stdp":
        out["weights"] = net.weights()
    if kind == "coba":
        # about 80 synapses per neuron, drawn: an array that holds any such network's
        w = net.weights()
        out["weights"] = np.zeros(96 * d.n_neurons, np.float32)
        out["weights"][:len(w)] = w
    return out


# Population rates these networks run at (Hz), from the settings above; they size work().
_RATE = {"groups": 40.0, "brunel": 43.0, "inputs": 30.0, "coba": 10.0, "stdp": 8.0, "large": 7.0, "plain": 0.0}


def work(case):
    """Bytes: 24 per neuron and step (membrane, refractory state, input slot; read and
    written), 16 per spike, 8 per delivery (target and weight), plus 24 per plastic update (the
    synapses of a spiking neuron, both sides) and what the caller reads; operations: 10 per
    neuron and step, one per delivery, the multiply-adds of the network for the surrogate."""
    kind = case["kind"]
    per_row = 2.0 * (5 * 256 + 3 * 256 * 256 + 256 * 3)
    if kind == "predict":
        r = case["members"] * case["rows"]
        return {"bytes": 20.0 * case["rows"] + 12.0 * r + 4.0 * mlp.PARAMS * case["members"], "flops": per_row * r}
    if kind == "train":
        r = case["members"] * case["batch"]
        p = 4.0 * mlp.PARAMS * case["members"]
        # a step reads and writes the weights and both moments, and reads its rows
        return {"bytes": (case["steps"] + 1) * (32.0 * r / case["members"] + 6 * p) + 3 * p,
                "flops": 3.0 * (case["steps"] + 1) * r * per_row}
    if kind in ("realise", "points"):
        # mean of the distribution: N log-uniform in 1250..12500, in-degree N / 10, ~40 Hz
        n, c, rate = 4900.0, 700.0, 40.0
        steps = case["seconds"] / 1e-4
        e = n * rate * case["seconds"] * c
        b = n * steps * 24 + n * rate * case["seconds"] * 16 + e * 8
        if kind == "points":
            b += n * c * 2   # the generated synapses, written once
        return {"bytes": case["points"] * b, "flops": case["points"] * (n * steps * 10 + e)}
    if kind == "plain":
        n, steps = 1000.0, float(case["groups"])
        e = 1000 * 20.0 * steps * 1e-4 * 100
        return {"bytes": 2 * n * steps * 24 + e * 8, "flops": 2 * n * steps * 10 + e}
    n = float(case["n"])
    if kind == "coba":
        steps, out, n_in, r_in, plastic = case["groups"] * 8.0, 80.0, 0.0, 0.0, 0.3
    elif kind in ("groups", "brunel"):
        steps, out, n_in, r_in, plastic = case["groups"] * float(case["delay"]), n / 10, 0.0, 0.0, 0.0
    elif kind == "inputs":
        steps, out, n_in, r_in, plastic = case["groups"] * float(case["delay"]), n / 10, 1e4, 20.0 * n / 1e4, 0.0
    else:
        k = float(case["out_degree"])
        steps, out, n_in, r_in, plastic = float(case["groups"]), k, n / 20, 10.0 * 1000 / k, 1.28
    t = steps * 1e-4
    spikes = n * _RATE[kind] * t + n_in * r_in * t
    e = spikes * out
    return {"bytes": (n + n_in) * steps * 24 + spikes * 16 + e * 8 + e * plastic * 24,
            "flops": n * steps * 10 + e + e * plastic * 10}


# ---- the surrogate in 64 bits -------------------------------------------------------------
# The simulations have no 64-bit value: a spike that a rounding moves by one step changes
# every later one.

_SHAPES = [(256, 5), (256,), (256, 256), (256,), (256, 256), (256,), (256, 256), (256,), (3, 256), (3,)]


def _split(flat):
    """[members][parameters] -> the five (W, b) pairs, batched over the members."""
    out, o = [], 0
    for s in _SHAPES:
        k = int(np.prod(s))
        out.append(flat[:, o:o + k].reshape(-1, *s))
        o += k
    return out


def _forward(flat, x):
    """y [members][rows][3] of x [members or 1][rows][5]."""
    p = _split(flat)
    a = x
    for k in range(4):
        a = torch.nn.functional.silu(torch.matmul(a, p[2 * k].transpose(1, 2).contiguous()) + p[2 * k + 1][:, None, :])
    return torch.matmul(a, p[8].transpose(1, 2).contiguous()) + p[9][:, None, :]


def _philox(block, member, stream, seed):
    """Philox4x32-10 (Salmon et al. 2011): the four words of each counter (block, member,
    stream) under key = seed, as uint64 arrays."""
    c = [block & 0xFFFFFFFF, block >> np.uint64(32), np.full_like(block, member), np.full_like(block, stream)]
    k0, k1 = seed & 0xFFFFFFFF, (seed >> 32) & 0xFFFFFFFF
    lo = np.uint64(0xFFFFFFFF)
    for _ in range(10):
        a, b = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(b >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), b & lo, (a >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), a & lo]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return c


def _sampled_rows(seed, step, batch, member, n):
    """The rows of one member's batch: draw step * batch + r of stream 4, scaled to [0, n)."""
    d = np.arange(step * batch, (step + 1) * batch, dtype=np.uint64)
    w = np.stack(_philox(d >> np.uint64(2), member, 4, seed))
    u = w[(d & np.uint64(3)).astype(np.int64), np.arange(batch)]
    return ((u * np.uint64(n)) >> np.uint64(32)).astype(np.int64)


def _loss_grads(flat, x, t):
    """Per-member loss (mean over rows of the summed squared error) and its gradient."""
    flat = flat.detach().requires_grad_(True)
    loss = (_forward(flat, x) - t).square().sum(2).mean(1)
    return loss.detach(), torch.autograd.grad(loss.sum(), flat)[0]


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    f64 = lambda a: torch.from_numpy(np.asarray(a, dtype=np.float64)).to(dev)
    if case["kind"] == "predict":
        p = f64(mlp.init_params(seed + 1, case["members"]))
        x = f64(np.random.default_rng(seed).uniform(-1.0, 1.0, (case["rows"], mlp.INPUTS)).astype(np.float32))
        return torch.cat([_forward(p, x[None, k:k + 65536]) for k in range(0, len(x), 65536)], 1).cpu().numpy()
    if case["kind"] != "train":
        return None
    x, t, p0 = _train_inputs(case, seed)
    n, m, b = case["data"], case["members"], case["batch"]
    x, t, p = f64(x), f64(t), f64(p0)
    rows = min(b, (n // mlp.ROW_TILE) * mlp.ROW_TILE)
    loss, grads = _loss_grads(p, x[None, :rows], t[None, :rows])
    mom, vel = torch.zeros_like(p), torch.zeros_like(p)
    for s in range(case["steps"]):
        idx = torch.from_numpy(np.stack([_sampled_rows(seed, s, b, e, n) for e in range(m)])).to(dev)
        _, g = _loss_grads(p, x[idx], t[idx])
        mom, vel = 0.9 * mom + 0.1 * g, 0.999 * vel + 0.001 * g * g
        p = p - _LR * (mom / (1 - 0.9 ** (s + 1))) / ((vel / (1 - 0.999 ** (s + 1))).sqrt() + 1e-8)
    return dict(loss=loss.cpu().numpy(), grads=grads.cpu().numpy(), params=p.cpu().numpy())
