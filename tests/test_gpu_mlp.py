"""GPU: BF16 MFMA MLP kernels against the NumPy oracle (forward, gradients),
and training reduces the loss."""
import ctypes as C

import numpy as np
import pytest

from oracle import mlp_oracle as MO

pytestmark = pytest.mark.gpu


def _net(nin=7, width=256, depth=4, nout=2, seed=11):
    import nosh_amd as nosh
    return nosh.Mlp(nin, width, depth, nout, seed)


@pytest.mark.parametrize("M", [64, 1000, 4096])
def test_forward_matches_oracle(M):
    net = _net()
    rng = np.random.default_rng(1)
    X = rng.normal(0, 1, (M, 7)).astype(np.float32)
    y = net.forward(X)
    p = net.get_params()
    y_bf, _, _ = MO.forward(p, X, net.dims, bf=True)
    err = np.linalg.norm(y - y_bf) / np.linalg.norm(y_bf)
    print("forward rel err vs bf16-emulating oracle", err)
    assert err < 5e-3
    y64, _, _ = MO.forward(p, X, net.dims, bf=False)
    assert np.linalg.norm(y - y64) / np.linalg.norm(y64) < 5e-2


def test_gradients_match_oracle():
    net = _net()
    rng = np.random.default_rng(2)
    M = 3000
    X = rng.normal(0, 1, (M, 7)).astype(np.float32)
    T = rng.normal(0, 1, (M, 2)).astype(np.float32)
    loss, g = net.gradients(X, T)
    p = net.get_params()
    loss_ref, g_ref = MO.loss_and_grad(p, X, T, net.dims, bf=True)
    assert abs(loss - loss_ref) / loss_ref < 5e-3
    # Layer by layer (weights, then biases).
    dims = net.dims
    off = 0
    for a, b in zip(dims[:-1], dims[1:]):
        s = slice(off, off + a * b)
        e = np.linalg.norm(g[s] - g_ref[s]) / np.linalg.norm(g_ref[s])
        print("weights", a, "x", b, "rel err", e)
        assert e < 2e-2
        off += a * b
    for b in dims[1:]:
        s = slice(off, off + b)
        e = np.linalg.norm(g[s] - g_ref[s]) / max(np.linalg.norm(g_ref[s]), 1e-30)
        assert e < 2e-2
        off += b


def test_training_reduces_loss():
    import torch
    net = _net(seed=3)
    rng = np.random.default_rng(4)
    M = 8192
    X = rng.uniform(-1, 1, (M, 7)).astype(np.float32)
    T = np.stack([np.sin(2 * X[:, 0]) * X[:, 1], X[:, 2] * X[:, 3] - 0.5 * X[:, 4]],
                 axis=1).astype(np.float32)
    dev = torch.device("cuda:0")
    Xd = torch.from_numpy(X).to(dev)
    Td = torch.from_numpy(T).to(dev)
    losses = [net.train_step_device(Xd.data_ptr(), Td.data_ptr(), M, 1e-3) for _ in range(300)]
    print("loss", losses[0], "->", losses[-1])
    assert losses[-1] < 0.1 * losses[0]


@pytest.mark.parametrize("width,depth,nin,M,nout", [
    (256, 4, 9, 1000, 2), (256, 2, 8, 16321, 16), (256, 2, 9, 32641, 5), (128, 3, 1, 300, 1),
    (128, 2, 32, 16384, 4), (128, 2, 5, 32768, 16), (64, 2, 9, 129, 5), (64, 1, 31, 20000, 16),
    (64, 4, 7, 32641, 3), (256, 1, 3, 33, 8), (128, 2, 7, 95, 13)])
def test_fused_inference_matches_forward(width, depth, nin, M, nout):
    """The one-kernel network gives the layer-by-layer path's values bit for
    bit (the same roundings in the same order of summation), at every number
    of rows a workgroup takes and in both forms of the last layer (up to four
    outputs and more). The layer-by-layer path is that of a network
    with more than 32 inputs: here the same network with 64 inputs of which
    those past the first n_in are zero, as are their weights, so that they add
    nothing. The two sum the gradients in orders of their own: their FP32 sums
    of some 500 rows at a time keep 1e-5 of sum |terms|, which is up to
    sqrt(M) = 180 times the gradient for targets without structure."""
    net = _net(nin=nin, width=width, depth=depth, nout=nout, seed=5)
    wide = _net(nin=64, width=width, depth=depth, nout=nout, seed=6)
    rng = np.random.default_rng(7)
    p = net.get_params()
    p[net.nweights:] = rng.uniform(-0.2, 0.2, net.nparams - net.nweights)
    net.set_params(p)

    def widen(v):
        first = np.zeros((width, 64), np.float32)
        first[:, :nin] = v[:width * nin].reshape(width, nin)
        return np.concatenate([first.ravel(), v[width * nin:]])

    wide.set_params(widen(p))
    X = rng.normal(0, 1, (M, nin)).astype(np.float32)
    Xw = np.concatenate([X, np.zeros((M, 64 - nin), np.float32)], axis=1)
    T = rng.normal(0, 1, (M, nout)).astype(np.float32)
    y = wide.forward(Xw)
    np.testing.assert_array_equal(wide.infer(Xw), y)
    np.testing.assert_array_equal(net.forward(X), y)
    np.testing.assert_array_equal(net.infer(X), y)
    loss, g = net.gradients(X, T)
    loss_w, g_w = wide.gradients(Xw, T)
    assert abs(loss - loss_w) <= 1e-12 * loss_w  # the same squares, summed in FP64
    assert np.linalg.norm(widen(g) - g_w) <= 2e-3 * np.linalg.norm(g_w)
    if M <= 1000:
        y_bf, _, _ = MO.forward(p, X, net.dims, bf=True)
        assert np.linalg.norm(y - y_bf) / np.linalg.norm(y_bf) < 5e-3


def test_first_adam_step_closed_form():
    """Adam's first step (beta1 0.9, beta2 0.999, eps 1e-8, bias-corrected)
    has a closed form: m_hat = g and v_hat = g^2, so every parameter moves by
    -lr g / (|g| + eps), i.e. -lr sign(g) where |g| >> eps. The step is
    checked against the gradient the library reports for the same minibatch
    (FP32 master weights: within a few ulps of the parameter)."""
    import torch
    net = _net(seed=5)
    rng = np.random.default_rng(6)
    M = 2048
    X = rng.normal(0, 1, (M, 7)).astype(np.float32)
    T = rng.normal(0, 1, (M, 2)).astype(np.float32)
    p0 = net.get_params().astype(np.float64)
    _, g = net.gradients(X, T)
    g = g.astype(np.float64)
    dev = torch.device("cuda:0")
    Xd = torch.from_numpy(X).to(dev)
    Td = torch.from_numpy(T).to(dev)
    lr = 1e-3
    net.train_step_device(Xd.data_ptr(), Td.data_ptr(), M, lr)
    torch.cuda.synchronize()
    d = net.get_params().astype(np.float64) - p0
    want = -lr * g / (np.abs(g) + 1e-8)
    tol = 4 * np.finfo(np.float32).eps * np.maximum(np.abs(p0), lr) + 1e-3 * lr
    assert np.all(np.abs(d - want) <= tol), np.max(np.abs(d - want) - tol)
    big = np.abs(g) > 1e-5
    assert big.sum() > 0.9 * g.size
    np.testing.assert_allclose(d[big], -lr * np.sign(g[big]), rtol=0, atol=2e-3 * lr + 1e-6)


@pytest.mark.parametrize("nin,width,depth,nout,M", [
    (1, 64, 1, 1, 1), (7, 64, 2, 2, 127), (10, 128, 3, 2, 128), (11, 128, 2, 3, 129),
    (21, 256, 2, 11, 257), (32, 256, 3, 16, 500), (9, 256, 4, 2, 40000), (5, 64, 2, 16, 63),
    (6, 256, 1, 3, 33), (7, 256, 2, 2, 16321), (7, 128, 2, 2, 16385), (7, 128, 2, 2, 32641),
    (7, 64, 2, 2, 32641)])
def test_fused_network_shapes(nin, width, depth, nout, M):
    """The fused kernels at the edges of their tiles: rows around the 32-, 64-
    and 128-row workgroups and the 512-row gradient splits, inputs around the
    32-column tiles of their three-part split (3 n_in + 1 = 31, 34, 64, 97), one
    hidden layer, and outputs on both sides of one 32-row tile of 3 n_out."""
    _check_against_oracle(nin, width, depth, nout, M)


@pytest.mark.parametrize("nin,width,depth,nout,M", [
    (7, 192, 3, 2, 1000), (40, 64, 2, 3, 500), (33, 128, 1, 1, 65), (64, 256, 2, 16, 127),
    (1, 320, 2, 2, 1), (9, 512, 2, 2, 1025)])
def test_layered_network_shapes(nin, width, depth, nout, M):
    """The layer-by-layer path of every other shape: widths without a fused
    kernel and more than 32 inputs, rows around its 64-row tiles, its 32-row
    reduction chunks and its 1024-row gradient splits."""
    _check_against_oracle(nin, width, depth, nout, M)


def _check_against_oracle(nin, width, depth, nout, M):
    net = _net(nin=nin, width=width, depth=depth, nout=nout, seed=9)
    rng = np.random.default_rng(12)
    p = net.get_params()
    p[net.nweights:] = rng.uniform(-0.2, 0.2, net.nparams - net.nweights)
    net.set_params(p)
    X = rng.normal(0, 1, (M, nin)).astype(np.float32)
    T = rng.normal(0, 1, (M, nout)).astype(np.float32)
    y_bf, _, _ = MO.forward(p, X, net.dims, bf=True)
    assert np.linalg.norm(net.infer(X) - y_bf) / np.linalg.norm(y_bf) < 5e-3
    loss, g = net.gradients(X, T)
    loss_ref, g_ref = MO.loss_and_grad(p, X, T, net.dims, bf=True)
    assert abs(loss - loss_ref) / loss_ref < 5e-3
    off = 0
    for size in [a * b for a, b in zip(net.dims[:-1], net.dims[1:])] + net.dims[1:]:
        s = slice(off, off + size)
        assert np.linalg.norm(g[s] - g_ref[s]) / np.linalg.norm(g_ref[s]) < 2e-2
        off += size
