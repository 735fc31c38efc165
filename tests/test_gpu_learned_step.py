"""The network's training iteration in sample tiles: gradients at the edges of its tiles (16 samples,
features padded to 32, the splits of the sample range) and on both sides of the rule that picks it, and
Adam's update with the BF16 copies it leaves, against the oracle."""
import os
import sys

import numpy as np
import pytest

from mcitest import ROOT

sys.path.insert(0, os.path.join(ROOT, "oracle"))
import mlp_oracle as M  # noqa: E402

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)


# the oracle rounds the products' operands to BF16 at the same places; an operand that falls on the
# other side of a rounding boundary (the sums' order differs) moves by one unit of 2^-8, so a gradient
# of few terms stays within 2^-7 of its norm; of many, few operands move (1e-5 to 3e-4 of the norm at
# 1,024 to 4,096 samples)
@pytest.mark.parametrize("d,H,K,n", [
    (1, 16, 1, 1),        # the smallest network, one sample
    (5, 40, 3, 17),       # padded inputs and hidden units, a ragged tile
    (33, 100, 2, 63),
    (32, 128, 8, 256),    # no split, two splits, many
    (32, 128, 8, 512),
    (16, 128, 8, 4099),
    (64, 128, 8, 80),     # outputs that just fit a compute unit
    (96, 128, 8, 70),     # and not: the products one by one
    (8, 1024, 2, 33),
])
def test_gradient_of_a_minibatch(d, H, K, n):
    from mcintegratorplusplus_amd.learned import Network
    print("network", d, H, K, n, flush=True)
    net = Network(d, H, K, seed=3)
    rng = np.random.default_rng(d + n)
    p = (net.params() + 0.05 * rng.normal(size=net.params().size)).astype(np.float32)  # biases too
    net.setParams(p)
    x = rng.normal(0.0, 2.0, (n, d)).astype(np.float32)
    y = (x + rng.normal(0.0, 1.0, (n, d))).astype(np.float32)
    loss, g = net.lossGrad(x, y)
    lo, go = M.loss_grad(p.astype(np.float64), x, y, d, H, K, emulate=True)
    assert abs(loss - lo) < 1e-3 * max(1.0, abs(lo))
    off = 0
    for name, shp in M.sizes(d, H, K):
        m = int(np.prod(shp))
        assert _rel(g[off:off + m], go[off:off + m]) < 2.0 ** -7, name
        off += m
    # a second, shorter minibatch in the same workspace
    n2 = (n + 1) // 2
    _, g2 = net.lossGrad(x[:n2], y[:n2])
    assert _rel(g2, M.loss_grad(p.astype(np.float64), x[:n2], y[:n2], d, H, K, emulate=True)[1]) < 2.0 ** -7


def test_training_leaves_the_copies_of_its_parameters():
    """after some iterations the network's own gradient (BF16 copies written by Adam) equals that of a
    network that is given the parameters (copies made from them)"""
    from mcintegratorplusplus_amd.learned import LearnedProposalSampler, Network, mixture_target
    d = 12
    w, mu, cov, _ = mixture_target(d=d, ncomp=3, seed=2)
    s = LearnedProposalSampler(w, mu, cov, 256)
    s.setSeed(5)
    s.setNetwork(72, 3)
    s.collect(4, 16)
    s.train(5, 100, 1e-3)
    net, other = s.network(), Network(d, 72, 3, seed=1)
    other.setParams(net.params())
    rng = np.random.default_rng(1)
    x = rng.normal(0.0, 2.0, (40, d)).astype(np.float32)
    a, b = net.lossGrad(x, x[::-1].copy()), other.lossGrad(x, x[::-1].copy())
    assert a[0] == b[0] and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("d,H,K,n", [
    (1, 800, 1, 48_000_000),   # sample tiles: 6.6 KB of workspace a sample, 316 GB
    (1, 1024, 1, 80_000_000),  # the products one by one: 4 KB a sample of the first layer's outputs, 328 GB
])
def test_a_minibatch_too_large_leaves_the_network_usable(d, H, K, n):
    """a workspace that cannot grow is an error, and later minibatches do not use what it held before"""
    from mcintegratorplusplus_amd.learned import Network
    print("workspace", d, H, K, n, flush=True)
    net = Network(d, H, K, seed=3)
    x = np.random.default_rng(1).normal(0.0, 2.0, (64, d)).astype(np.float32)
    loss, g = net.lossGrad(x, x[::-1].copy())
    big = np.zeros((n, d), np.float32)
    with pytest.raises(RuntimeError):
        net.lossGrad(big, big)
    l2, g2 = net.lossGrad(x, x[::-1].copy())
    assert l2 == loss and np.array_equal(g, g2)
