"""The surrogate's inference over the sizes at which another kernel or tile takes over (16-row
tiles, 64-row tiles, 128-row tiles, pieces copied while the next computes): every row's outputs
are those of a call of another size, bit for bit, and those of the FP64 restatement
(oracle/mlp_oracle.py, relative L2 1e-3 against its BF16 mode as in test_gpu_mlp); parameters
that are not finite are refused and leave the current ones in place."""
import numpy as np
import pytest

import mlp_oracle as mo
from spike_amd import abi, mlp
from test_gpu_mlp import rel, rows

pytestmark = pytest.mark.gpu


def _check(models, sizes):
    params = mlp.init_params(5, models)
    m = mlp.Mlp(models, 128)
    m.set_params(params)
    x, _ = rows(6, max(sizes))
    whole = m.predict(x)
    check = np.unique(np.concatenate([np.arange(40), np.random.default_rng(2).choice(len(x), 200), np.arange(len(x) - 40, len(x))]))
    for e in range(models):
        assert rel(whole[e][check], mo.forward(params[e], x[check], mode="bf16")[0]) <= 1e-3
    for n in sizes[:-1]:
        print("rows", n, flush=True)
        assert np.array_equal(m.predict(x[:n]), whole[:, :n]), n
        assert np.array_equal(m.predict(x[len(x) - n:]), whole[:, len(x) - n:]), n
    m.close()


def test_one_member():
    _check(1, [1, 15, 16, 17, 63, 64, 65, 4095, 4096, 4097, 65535, 65537, 131071, 131072, 131073, 200001])


def test_eight_members():
    _check(8, [1, 31, 100, 511, 512, 513, 8191, 8193, 16383, 16384, 16385, 40001])


def test_sixty_four_members():
    _check(64, [1, 16, 63, 64, 65, 1023, 1025, 2047, 2048, 2049, 5003])


def test_training_tiles():
    """A batch in 128-row tiles (over 256 of them) against its halves in 64-row tiles: the
    gradient of a batch is the mean of its halves' gradients (FP32 sums in another order)."""
    params = mlp.init_params(7, 7)
    x, t = rows(8, 8192)
    g = []
    for part in (slice(None), slice(0, 4096), slice(4096, None)):
        m = mlp.Mlp(7, 8192)
        m.set_params(params)
        m.set_data(x[part], t[part])
        g.append(m.gradients(len(x[part])))
        m.close()
    for e in range(7):
        assert abs(g[0][0][e] - 0.5 * (g[1][0][e] + g[2][0][e])) <= 1e-5 * g[0][0][e]
        assert rel(g[0][1][e], 0.5 * (np.asarray(g[1][1][e], np.float64) + g[2][1][e])) <= 1e-5


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_parameters_that_are_not_finite(bad):
    params = mlp.init_params(9, 2)
    m = mlp.Mlp(2, 128)
    m.set_params(params)
    x, _ = rows(10, 50)
    y = m.predict(x)
    wrong = params.copy()
    wrong[1, -1] = bad
    wrong[0, 4711] = bad
    with pytest.raises(abi.SpikeError, match="non-finite parameter at 4711"):
        m.set_params(wrong)
    assert np.array_equal(m.predict(x), y) and np.array_equal(m.params(), params)
    m.close()
