"""The order of the network's FP32 sums, to the bit: an output adds its columns
tile after tile of 16, then over the 16 columns of a tile; a workgroup's weight
gradients, its last bias's and its loss are those of its 16-row tiles added one
after the other, its columns' gradients those of its 4-row groups; the
workgroups follow in order.  A step on a power of two of rows scales exactly with that number, so
the parts come from calls of their own."""
import numpy as np
import pytest

from oracle import mlp as omlp

pytestmark = pytest.mark.gpu

TILES = [slice(omlp.OFF_W1, omlp.OFF_B1), slice(omlp.OFF_W2, omlp.OFF_B2), slice(omlp.OFF_B3, omlp.NPARAM)]
COLUMNS = [slice(omlp.OFF_B1, omlp.OFF_W2), slice(omlp.OFF_B2, omlp.OFF_B3)]


def rows_of(n, seed):
    rng = np.random.default_rng(seed)
    return rng.normal(size=(n, 16)).astype(np.float32), rng.normal(size=n).astype(np.float32)


def summed(net, x, t, part):
    """Gradient and loss of the rows as the parts' own, added in FP32 in their order."""
    n = len(t)
    g, s = np.zeros(omlp.NPARAM, np.float32), np.float32(0)
    for k in range(0, n, part):
        gk, lk = net.gradients(x[k:k + part], t[k:k + part])
        g = g + gk * np.float32(part / n)
        s = s + np.float32(lk) * np.float32(part)
    return g, s / np.float32(n)


@pytest.mark.parametrize("seed", [1, 2])
def test_tiles_of_a_workgroup(seed):
    from sassena_amd.mlp import MLP
    x, t = rows_of(64, seed)
    with MLP(seed=seed) as net:
        g, loss = net.gradients(x, t)
        g16, l16 = summed(net, x, t, 16)
        g4, _ = summed(net, x, t, 4)
    for s in TILES:
        assert np.array_equal(g[s], g16[s]), s
    for s in COLUMNS:
        assert np.array_equal(g[s], g4[s]), s
    assert np.float32(loss) == l16


@pytest.mark.parametrize("rows", [128, 4096, 8192])
def test_workgroups(rows):
    from sassena_amd.mlp import MLP
    x, t = rows_of(rows, rows)
    with MLP(seed=3) as net:
        g, loss = net.gradients(x, t)
        g64, l64 = summed(net, x, t, 64)
    assert np.array_equal(g, g64)
    assert np.float32(loss) == l64


def test_output_of_a_row():
    from sassena_amd.mlp import MLP
    rng = np.random.default_rng(4)
    p = np.zeros(omlp.NPARAM, np.float32)
    sign = rng.choice([-1.0, 1.0], size=128).astype(np.float32)
    p[omlp.OFF_B2:omlp.OFF_W3] = 100.0 * sign  # tanh is exactly +-1
    w3 = rng.normal(size=128).astype(np.float32)
    p[omlp.OFF_W3:omlp.OFF_B3] = w3
    p[omlp.OFF_B3] = np.float32(0.3)
    s = np.zeros(16, np.float32)
    for tile in range(8):
        s = s + (sign * w3)[16 * tile:16 * tile + 16]
    for off in (8, 4, 2, 1):
        s = s + s[np.arange(16) ^ off]
    with MLP(seed=1) as net:
        net.set_params(p)
        y = net.predict(rows_of(70, 5)[0])
    assert np.all(y == s[0] + np.float32(0.3)), (y[0], s[0])
