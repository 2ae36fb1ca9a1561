"""Network products at the edges of their tiles (16 and 32 wide), of the chunks
along the contraction (32) and of the waves that share them (8): widths of 1,
odd widths, rows around 16, against the FP64 oracle with BF16 operands."""
import numpy as np
import pytest

from oracle import mlp as OM

pytestmark = pytest.mark.gpu


def _net(dims, seed):
    from cfft_hip.mlp import MLP
    net = MLP(dims, seed=seed)
    p = net.params()
    p[-sum(dims[1:]):] = np.random.default_rng(seed).standard_normal(sum(dims[1:])).astype(np.float32)
    net.set_params(p)
    return net, p


@pytest.mark.parametrize("K,N,rows", [(1, 1, 1), (1, 7, 17), (5, 1, 16), (2, 2, 33), (31, 17, 15), (32, 32, 32),
                                      (33, 35, 31), (200, 31, 65), (257, 33, 100), (290, 16, 300)])
def test_one_layer(K, N, rows):
    """One linear layer: the operands are the oracle's own BF16 values, so the
    output differs by FP32 sums of K terms only.  The output gradient may round
    to the other BF16 neighbour: 2^-8 of each term of the weight gradient."""
    net, p = _net([K, N], 7)
    rng = np.random.default_rng(K + N + rows)
    x = rng.standard_normal((rows, K)).astype(np.float32)
    t = rng.standard_normal((rows, N)).astype(np.float32)
    xb, wb = OM.bf16(x).astype(float), OM.bf16(p[:K * N]).astype(float).reshape(K, N)
    b = p[K * N:].astype(float)
    y = xb @ wb + b
    ytol = (K + 4) * 2.0 ** -23 * (np.abs(xb) @ np.abs(wb) + np.abs(b))
    assert np.all(np.abs(net.forward(x) - y) <= ytol)
    loss, g = net.gradient(x, t)
    d = y - t
    dy, dtol = 2 * d / d.size, 2 * (ytol + 2.0 ** -22 * np.abs(d)) / d.size
    assert abs(loss - np.mean(d * d)) <= np.mean(2 * np.abs(d) * ytol + ytol ** 2) + 2.0 ** -23 * np.mean(d * d)
    wtol = np.abs(xb).T @ (np.abs(dy) * (2.0 ** -7 + (rows + 4) * 2.0 ** -23) + 2 * dtol)
    assert np.all(np.abs(g[:K * N].reshape(K, N) - xb.T @ OM.bf16(dy.astype(np.float32)).astype(float)) <= wtol)
    btol = (dtol + (rows + 4) * 2.0 ** -23 * np.abs(dy)).sum(0)
    assert np.all(np.abs(g[K * N:] - dy.sum(0)) <= btol)


@pytest.mark.parametrize("dims,rows", [([3, 1, 2], 5), ([6, 17, 33, 5], 33), ([6, 64, 31, 256], 1),
                                       ([2, 290, 45, 3], 47), ([6, 200, 200, 200, 256], 513)])
def test_layers(dims, rows):
    """Several layers: an activation that rounds the other way moves what
    follows by up to 2^-8 of it, two roundings per layer deep."""
    net, p = _net(dims, 11)
    rng = np.random.default_rng(rows)
    x = rng.standard_normal((rows, dims[0])).astype(np.float32)
    t = rng.standard_normal((rows, dims[-1])).astype(np.float32)
    yr = OM.forward(p, dims, x)[0][-1]
    assert np.linalg.norm(net.forward(x) - yr) <= 2.0 ** -6 * np.linalg.norm(yr)
    loss, g = net.gradient(x, t)
    lr, gr = OM.loss_and_grad(p, dims, x, t)
    assert abs(loss - lr) <= 2.0 ** -6 * lr
    off = 0
    for n in [a * b for a, b in zip(dims[:-1], dims[1:])] + dims[1:]:
        assert np.linalg.norm(g[off:off + n] - gr[off:off + n]) <= 2.0 ** -6 * np.linalg.norm(gr[off:off + n])
        off += n


def test_refused_allocation_is_reported_once():
    """A batch whose activations cannot be allocated (15 TB) is refused on the
    host; the next launches, of another object, do not report it again."""
    import cfft_hip as cf
    net, _ = _net([6, 512, 512, 512, 256], 13)
    x, t = np.ones((8, 6), np.float32), np.ones((8, 256), np.float32)
    N = (32, 32, 32)
    _, ops_s = cf.find_optimal_shift(cf.get_ops(229, 3, N), N)
    plan = cf.DevicePlan(N, ops_s, 0.01, 4.0 * np.eye(3), cf.PATH_M7, cf.FP64)
    f = np.random.default_rng(3).standard_normal(plan.M)
    want = plan.diffuse(f)
    with pytest.raises(cf.CFFTError) as e:
        net.train(x, t, epochs=1, batch=2 ** 31 - 1)
    assert e.value.code == cf._lib.CFFT_ERR_HIP
    assert np.array_equal(plan.diffuse(f), want)


def test_failed_allocation_leaves_the_network_usable():
    """A batch whose activations cannot be allocated (15 TB) is refused on the
    host; the calls after it allocate their own and compute as before."""
    import cfft_hip as cf
    dims = [6, 512, 512, 512, 256]
    net, _ = _net(dims, 13)
    rng = np.random.default_rng(13)
    x = rng.standard_normal((8, 6)).astype(np.float32)
    t = rng.standard_normal((8, 256)).astype(np.float32)
    loss, g = net.gradient(x, t)
    with pytest.raises(cf.CFFTError) as e:
        net.train(x, t, epochs=1, batch=2 ** 31 - 1)
    assert e.value.code == cf._lib.CFFT_ERR_HIP
    loss2, g2 = net.gradient(x, t)
    assert loss2 == loss and np.array_equal(g2, g)
