"""GPU: the whole-network surrogate kernels (pm_mlp_net_*) at the edges of
their tiles: widths that are not multiples of 16 or 32, up to the 512 limit,
one to a few hundred rows, both workgroup heights.

Layer by layer against O2 fed the device's own inputs, as the per-layer GEMM
tests: FP32 sums of BF16 products, bar 1e-5 (max-norm).  A minibatch's
gradients against ``SpectralMLP.backward``, which takes one GEMM per layer and
is itself pinned against O2, at the same bar.
"""

import numpy as np
import pytest

from tests.test_gpu_mlp import _rel, _t

pytestmark = pytest.mark.gpu


def _net(n_in, hidden, depth, n_out, seed=3):
    from prismo_amd.surrogate.mlp import SpectralMLP

    net = SpectralMLP(n_in=n_in, n_out=n_out, hidden=hidden, depth=depth, seed=seed)
    rng = np.random.default_rng(seed)
    for b in net.b:
        b.copy_(_t(rng.normal(0, 0.1, b.shape)))
    return net


@pytest.mark.parametrize("M,n_in,hidden,depth,n_out", [
    (1, 4, 16, 1, 1), (15, 1, 33, 2, 45), (17, 4, 100, 3, 20), (130, 7, 256, 4, 256),
    (37, 40, 257, 2, 320), (20, 4, 512, 2, 512), (64, 33, 64, 11, 17)])
def test_forward_layers(mi355x, M, n_in, hidden, depth, n_out):
    from oracle import mlp as O2

    net = _net(n_in, hidden, depth, n_out)
    assert net._net() is not None
    X = _t(np.random.default_rng(M).uniform(-1, 1, (M, n_in)))
    Y, (acts, zs) = net.forward(X, keep=True)
    assert len(acts) == depth + 2 and len(zs) == depth and acts[-1] is Y
    P = net.params()
    for k, (W, b) in enumerate(P):
        z = O2.bf16(acts[k].cpu().numpy()) @ O2.bf16(W).T + b
        if k < depth:
            zk = zs[k].cpu().numpy()
            assert _rel(zk, z) <= 1e-5, k
            assert _rel(acts[k + 1].cpu().numpy(), O2.gelu(zk.astype(np.float64))) <= 1e-5, k
        else:
            assert _rel(Y.cpu().numpy(), z) <= 1e-5


@pytest.mark.parametrize("M,hidden", [(70, 40), (3000, 256), (300, 520)])
def test_activations_are_those_of_erf(mi355x, M, hidden):
    """Hidden values are z (1 + erf(z / sqrt 2)) / 2 in FP32 to the last bit, in the
    whole-network kernels and in the per-layer ones (520 units): one bit more or
    less turns some of their BF16 roundings, 2^-9 each, and the outputs with them."""
    import torch

    net = _net(4, hidden, 3, 8)
    X = _t(np.random.default_rng(1).uniform(-3, 3, (M, 4)))
    _, (acts, zs) = net.forward(X, keep=True)
    for k, z in enumerate(zs):
        assert torch.equal(acts[k + 1], 0.5 * z * (1.0 + torch.erf(z * 0.70710678118654752))), k


@pytest.mark.parametrize("hidden,n_out", [(40, 30), (128, 100), (256, 256), (300, 64)])
def test_tall_and_short_workgroups_agree(mi355x, hidden, n_out):
    """Enough rows for 128- (or 64-) row workgroups, with a ragged last one,
    against the same rows in small calls: the same products in the same order,
    so the same bits."""
    import torch

    net = _net(4, hidden, 3, n_out)
    M = 256 * 128 + 77
    X = _t(np.random.default_rng(1).uniform(-1, 1, (M, 4)))
    big = net.forward(X)
    for r0 in (0, 5000, M - 100):
        assert torch.equal(big[r0:r0 + 100], net.forward(X[r0:r0 + 100])), r0


@pytest.mark.parametrize("M,batch,hidden,depth,n_out,wd", [
    (40, 64, 48, 3, 12, 0.0), (100, 33, 100, 2, 45, 0.0), (65, 16, 256, 4, 64, 0.01),
    (50, 50, 300, 1, 20, 0.0)])
def test_training_matches_layer_calls(mi355x, M, batch, hidden, depth, n_out, wd):
    """fit() for one epoch against the same minibatches through forward, mse,
    backward and adam_step; weighted loss; the gradients of the last
    minibatch and the parameters."""
    rng = np.random.default_rng(7)
    X = _t(rng.uniform(-1, 1, (M, 4)))
    T = _t(rng.normal(size=(M, n_out)))
    w = _t(rng.uniform(0.5, 2.0, n_out))
    a, b = _net(4, hidden, depth, n_out), _net(4, hidden, depth, n_out)
    hist = a.fit(X, T, epochs=1, batch=batch, lr=1e-3, w=w, seed=5, wd=wd)
    perm = np.random.default_rng(5).permutation(M)
    nb = (M + batch - 1) // batch
    tot = 0.0
    for s in range(nb):
        i = perm[s * batch:(s + 1) * batch]
        Y, cache = b.forward(X[i], keep=True)
        loss, dY = b.mse(Y, T[i], w)
        grads = b.backward(cache, dY)
        lr = 1e-4 + 0.5 * (1e-3 - 1e-4) * (1 + np.cos(np.pi * s / nb))
        b.adam_step(grads, lr=float(lr), wd=wd)
        tot += loss.item()
    assert abs(hist[0] - tot / nb) <= 1e-5 * abs(hist[0])
    assert a.t == b.t == nb
    for k in range(depth + 1):
        assert _rel(a._gW[k].cpu().numpy(), grads[k][0].cpu().numpy()) <= 1e-5, k
        assert _rel(a._gb[k].cpu().numpy(), grads[k][1].cpu().numpy()) <= 1e-5, k
        assert _rel(a.W[k].cpu().numpy(), b.W[k].cpu().numpy()) <= 1e-5, k


@pytest.mark.parametrize("members,M,n_out", [(1, 3, 5), (2, 7, 33), (5, 600, 256)])
def test_predict_statistics(mi355x, members, M, n_out):
    from prismo_amd.surrogate.mlp import SurrogateEnsemble

    ens = SurrogateEnsemble(n_members=members, n_in=4, n_out=n_out, hidden=32, depth=2)
    X = _t(np.random.default_rng(2).uniform(-1, 1, (M, 4)))
    mean, std = ens.predict(X)
    S = np.stack([m.forward(X).cpu().numpy() for m in ens.members]).astype(np.float64)
    assert _rel(mean.cpu().numpy(), S.mean(0)) <= 1e-6
    if members == 1:
        assert bool(std.isnan().all())
    else:
        assert _rel(std.cpu().numpy(), S.std(0, ddof=1)) <= 1e-5


def test_networks_the_kernels_do_not_take(mi355x):
    """Wider than 512 units: the per-layer path, as before."""
    net = _net(4, 520, 1, 8)
    assert net._net() is None
    X = _t(np.random.default_rng(2).uniform(-1, 1, (9, 4)))
    Y, (acts, zs) = net.forward(X, keep=True)
    assert Y.shape == (9, 8) and zs[0].shape == (9, 520)
    assert len(net.fit(X, Y * 0, epochs=2, batch=4)) == 2
