"""The network's step at the edges of its 16-row tiles, 64-row workgroups and
the 16 slices that sum them, against the FP64 oracle; and the operand fragments
after training."""
import numpy as np
import pytest

from oracle import mlp as omlp

pytestmark = pytest.mark.gpu

# BF16 roundings of an activation that FP32 and FP64 put on different sides of a
# tie: 2^-8 of one of 128, well below this in the norm of a block of parameters
TOL = 2e-3


@pytest.mark.parametrize("rows", [1, 15, 17, 63, 65, 129, 1024, 1090])
def test_gradients(rows):
    from sassena_amd.mlp import MLP
    rng = np.random.default_rng(rows)
    x = rng.normal(size=(rows, 16)).astype(np.float32)
    t = rng.normal(size=rows).astype(np.float32)
    with MLP(seed=4) as net:
        p = net.params()
        g, loss = net.gradients(x, t)
        y = net.predict(x)
    p64 = p.astype(np.float64)
    rg, rloss = omlp.grads(p64, x.astype(np.float64), t.astype(np.float64))
    assert abs(loss - rloss) <= 1e-4 * rloss
    for a, b in ((omlp.OFF_W1, omlp.OFF_B1), (omlp.OFF_B1, omlp.OFF_W2), (omlp.OFF_W2, omlp.OFF_B2),
                 (omlp.OFF_B2, omlp.OFF_W3), (omlp.OFF_W3, omlp.OFF_B3), (omlp.OFF_B3, omlp.NPARAM)):
        assert np.linalg.norm(g[a:b] - rg[a:b]) < TOL * np.linalg.norm(rg[a:b]), (a, b)
    # the prediction and the loss come from the same forward pass, the loss summed in FP32
    assert abs(np.mean((y.astype(np.float64) - t) ** 2) - loss) <= 1e-4 * loss


@pytest.mark.parametrize("batch", [1, 70, 300])
def test_training_is_reproducible_and_refreshes_the_operands(batch):
    from sassena_amd.mlp import MLP
    rng = np.random.default_rng(batch)
    x = rng.normal(size=(500, 16)).astype(np.float32)
    t = np.tanh(x[:, 0]).astype(np.float32)
    out = []
    for _ in range(2):
        with MLP(seed=2) as net:
            loss = net.train(x, t, steps=20, batch=batch)
            out.append((net.params(), loss, net.predict(x)))
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]
    with MLP(seed=3) as net:
        net.set_params(out[0][0])
        assert np.array_equal(net.predict(x), out[0][2])
