"""Several training steps of the MLP kernels, and the row kernels' products
against the layer GEMM (fg_bf16_gemm), bit for bit."""
import ctypes
import ctypes.util

import numpy as np
import pytest

from cudaprotoplanetarydisks_amd.mlp import MLP, bf16_gemm

pytestmark = pytest.mark.gpu

F = np.float32


def powf(x, n):
    libm = ctypes.CDLL(ctypes.util.find_library("m"))
    libm.powf.restype = ctypes.c_float
    return F(libm.powf(ctypes.c_float(x), ctypes.c_float(n)))


@pytest.mark.parametrize("widths, batch", [([130, 129, 300, 9], 37), ([5, 70, 33, 45], 64), ([7, 20], 5), ([5, 900, 7], 20)])
def test_steps_over_two_batches(widths, batch):
    """Four Adam steps over two batches.  Each step, taken alone, from the
    parameters the last one left: its loss and its gradients are those that a
    network set to these parameters forms (whose weight copies are made anew), bit
    for bit, and the new parameters follow from them by Adam with the moments of
    all steps so far.  The moments take additions and products only, the same in
    numpy; the update's root and quotients are within an ulp each: 2^-20 of the
    step, and the subtraction an ulp of the parameter.  The four steps in one call
    give the same losses and parameters."""
    rng = np.random.default_rng(batch)
    x = rng.uniform(-1, 1, size=(2 * batch, widths[0])).astype(F)
    t = rng.normal(size=(2 * batch, widths[-1])).astype(F)
    lr, b1, b2, eps, steps = F(1e-2), F(0.9), F(0.999), F(1e-8), 4
    with MLP(widths, max_batch=batch, seed=11) as net, MLP(widths, max_batch=batch, seed=12) as fresh:
        p = net.params().astype(F)
        m, v = np.zeros_like(p), np.zeros_like(p)
        losses = []
        for s in range(steps):
            rows = slice(s % 2 * batch, (s % 2 + 1) * batch)
            fresh.set_params(p)
            loss, g = fresh.gradient(x[rows], t[rows])
            losses.append(net.train(x[rows], t[rows], batch=batch, steps=1, lr=lr)[0])
            assert losses[s] == loss, s
            g = g.astype(F)
            m = b1 * m + (F(1) - b1) * g
            v = b2 * v + (F(1) - b2) * g * g
            c1, c2 = F(1) - powf(b1, s + 1), F(1) - powf(b2, s + 1)
            step = lr * (m / c1) / (np.sqrt(v / c2) + eps)
            got = net.params().astype(F)
            excess = np.abs(got.astype(float) - (p - step)) - (2.0 ** -20 * np.abs(step) + 2.0 ** -23 * np.abs(p))
            assert excess.max() <= 0.0, (s, excess.max())
            p = got
    with MLP(widths, max_batch=batch, seed=11) as net:
        assert np.array_equal(net.train(x, t, batch=batch, steps=steps, lr=lr), losses)
        assert np.array_equal(net.params().astype(F), p)


@pytest.mark.parametrize("K, N, batch", [(5, 48, 1), (130, 300, 100), (257, 33, 37), (896, 130, 65)])
def test_products_are_the_layer_gemms(K, N, batch):
    """One dense layer: output, weight and bias gradient are what the layer
    GEMM, an FP32 addition of the bias and a sum over the rows in order give."""
    rng = np.random.default_rng(K)
    x = rng.normal(size=(batch, K)).astype(F)
    t = rng.normal(size=(batch, N)).astype(F)
    with MLP([K, N], max_batch=batch, seed=3) as net:
        p = rng.normal(size=net.nparam).astype(F)
        net.set_params(p)
        y = net.forward(x).astype(F)
        _, g = net.gradient(x, t)
    W, b = p[:N * K].reshape(N, K), p[N * K:]
    assert np.array_equal(y, bf16_gemm(x, W.T) + b)
    dz = F(2) / F(batch * N) * (y - t)
    assert np.array_equal(g[:N * K].reshape(N, K).astype(F), bf16_gemm(dz.T, x))
    assert np.array_equal(g[N * K:].astype(F), np.cumsum(dz, axis=0, dtype=F)[-1])


@pytest.mark.parametrize("M, N, batch", [(48, 5, 1), (300, 130, 100), (33, 257, 37), (130, 896, 65)])
def test_way_back_is_the_layer_gemm(M, N, batch):
    """Two layers with zero input and biases, where GELU' is 1/2 exactly: the
    first layer's bias gradient is half the layer GEMM of the output's gradients
    and the second weights, summed over the rows in order."""
    rng = np.random.default_rng(M)
    t = rng.normal(size=(batch, N)).astype(F)
    K = 3
    with MLP([K, M, N], max_batch=batch, seed=3) as net:
        W = rng.normal(size=(N, M)).astype(F)
        p = np.concatenate([rng.normal(size=M * K), np.zeros(M), W.ravel(), np.zeros(N)]).astype(F)
        net.set_params(p)
        _, g = net.gradient(np.zeros((batch, K)), t)
    dz = F(2) / F(batch * N) * (F(0) - t)
    below = F(0.5) * bf16_gemm(dz, W)
    assert np.array_equal(g[M * K:M * K + M].astype(F), np.cumsum(below, axis=0, dtype=F)[-1])
