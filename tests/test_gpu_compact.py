"""Networks whose sources weigh as one of two values (2-byte delivery records), bit-exact
against the FP32 oracle: the range of sources with the second value in the middle, at either
end, empty or of one source, inputs weighing as either, and a third range (full records)."""
import numpy as np
import pytest

import oracle_py
from spike_amd import abi, builders
from test_gpu_parity import _compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("partitions", [0, 3])
@pytest.mark.parametrize("n_inputs", [37, 301])
@pytest.mark.parametrize("hi,record_bytes", [((70, 97), 2), ((97, 400), 2), ((0, 20), 2), ((40, 41), 2), ((0, 0), 2),
                                             ((60, 110), 2), ((10, 20, 30, 40), 8), ((0, 10, 20, 30), 8)])
def test_two_weights(hi, record_bytes, n_inputs, partitions):
    d = builders.random_net(n_neurons=97, n_inputs=n_inputs, p=0.2, seed=7, dmin=6, dmax=6, input_rate=300.0)
    u = np.where(d.pre >= 0, d.pre, 97 - d.pre.astype(np.int64) - 1)
    is_hi = np.zeros(len(u), bool)
    for a, b in zip(hi[::2], hi[1::2]):
        is_hi |= (u >= a) & (u < b)
    d.weight = np.where(is_hi, np.float32(-2.5e-3), np.float32(1.5e-3)).astype(np.float32)
    gpu = abi.Network(d, partitions=partitions)
    ora = oracle_py.OracleNetwork(d, precision=32)
    assert gpu.info().fused == 1 and gpu.info().record_bytes == record_bytes
    t = 0.0
    for ng in (60, 1, 25):
        gpu.run(t, ng)
        ora.run(t, ng)
        t = float(d.group_time(t, ng))
        _compare(gpu, ora, d)
