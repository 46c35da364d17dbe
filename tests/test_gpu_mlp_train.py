"""Training kernel of the preconditioner network at its tile and block edges: 16-sample
tiles, four tiles per block, at most 256 blocks (more samples: several tiles per wave)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 16384, 16385, 20011])
def test_loss_and_gradient_at_tile_edges(n):
    print(f"mlp loss_grad n={n}", flush=True)
    import mlp as OM
    from hpmp.learned import MLP
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, 11)).astype(np.float32)
    T = rng.standard_normal((n, 9)).astype(np.float32)
    net = MLP(n)
    w = net.weights()
    w += 0.02 * rng.standard_normal(w.size).astype(np.float32)   # biases included
    net.set_weights(w)
    loss, g = net.loss_grad(X, T)
    lo, go = OM.loss_and_grad(w, X, T)
    # an activation that rounds the other way to bfloat16 (tanhf's last bit) moves by 2^-8
    # of itself; FP32 sums are far below that
    assert abs(loss - lo) <= 2.0 ** -8 * abs(lo)
    for a, b in ((0, 704), (704, 768), (768, 4864), (4864, 4928), (4928, 9024), (9024, 9088), (9088, 9664), (9664, 9673)):
        assert np.linalg.norm(g[a:b] - go[a:b]) <= 2.0 ** -8 * np.linalg.norm(go[a:b])


def test_epoch_loss_is_the_sample_mean_over_ragged_minibatches():
    import mlp as OM
    from hpmp.learned import MLP
    rng = np.random.default_rng(3)
    X = rng.standard_normal((200, 11)).astype(np.float32)
    T = rng.standard_normal((200, 9)).astype(np.float32)
    net = MLP(5)
    w = net.weights()
    last = net.train(X, T, epochs=1, batch=256, lr=0.0)
    lo, _ = OM.loss_and_grad(w, X, T)
    assert abs(last - lo) <= 2.0 ** -8 * abs(lo)
    assert np.array_equal(net.weights(), w)
    # 128 + 72 samples with a zero step: the epoch loss is the sample mean
    assert abs(net.train(X, T, epochs=2, batch=128, lr=0.0) - lo) <= 2.0 ** -8 * abs(lo)


@pytest.mark.parametrize("n", [1 << 18, (1 << 20) + 5])
def test_loss_of_a_large_minibatch_keeps_its_digits(n):
    """A network of zeros against one target value: every squared difference is the same
    FP32 number v, and the mean of n x 9 of them (at most 24 + 24 bits in the sum) is v."""
    print(f"mlp loss n={n}", flush=True)
    from hpmp.learned import MLP
    X = np.random.default_rng(1).standard_normal((n, 11)).astype(np.float32)
    T = np.full((n, 9), 0.123, np.float32)
    net = MLP(1)
    net.set_weights(np.zeros_like(net.weights()))
    v = float(np.float32(0.123) * np.float32(0.123))
    loss, _ = net.loss_grad(X, T)
    assert loss == v
    assert net.train(X, T, epochs=1, batch=n, lr=0.0) == v
