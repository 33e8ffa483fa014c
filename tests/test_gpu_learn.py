"""The early-stop network's device kernels against the CPU oracle
(oracle/convnet.py): forward pass, loss gradient and Adam steps (one with
a clipped gradient), on
the same parameters and inputs. The device accumulates in f32 in its own
order (multiply-adds contracted), so values agree to a tolerance: 2e-5 of
the largest magnitude for outputs, 2e-4 for gradients and 1e-5 for
parameters after a step."""
import ctypes as C

import numpy as np
import pytest

from ems_amd import _native as nat
from oracle import convnet as O

pytestmark = pytest.mark.gpu


def _net(cin, cout, ch, dil, seed):
    from ems_amd.learn import ConvNet
    return ConvNet(cin, cout, ch, dil, seed=seed)


def _close(a, b, tol):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    scale = max(np.abs(b).max(), 1e-30)
    err = np.abs(a - b).max() / scale
    assert err <= tol, f"max error {err:.3e} of the largest magnitude {scale:.3e}"


@pytest.mark.parametrize("shape", [(4, 2, 64, (1, 2, 4, 8, 16, 32), 2, 512),
                                   (3, 1, 16, (1, 3), 3, 37),
                                   (2, 3, 8, (2, 1, 5), 1, 1)])
def test_forward_matches_oracle(shape):
    cin, cout, ch, dil, B, T = shape
    n = _net(cin, cout, ch, dil, 1)
    p = n.params()
    s = O.Shape(cin, cout, ch, dil)
    assert p.size == s.count
    rng = np.random.default_rng(4)
    x = rng.standard_normal((B, cin, T)).astype(np.float32)
    got = n.forward(x)
    want = O.forward(s, p.astype(np.float64), x.astype(np.float64))
    _close(got, want, 2e-5)
    n.close()


@pytest.mark.parametrize("t0", [0, 100])
def test_gradient_matches_oracle(t0):
    dil = (1, 2, 4, 8, 16, 32)
    n = _net(4, 2, 64, dil, 7)
    s = O.Shape(4, 2, 64, dil)
    rng = np.random.default_rng(t0 + 1)
    # non-trivial parameters: perturb the initial ones, biases too
    p = n.params() + rng.standard_normal(s.count).astype(np.float32) * 0.02
    n.set_params(p)
    x = rng.standard_normal((3, 4, 256)).astype(np.float32)
    y = rng.standard_normal((3, 2, 256)).astype(np.float32)
    loss, g = n.loss_grad(x, y, t0)
    lo, go = O.loss_and_grad(s, p.astype(np.float64), x.astype(np.float64), y.astype(np.float64), t0)
    assert abs(loss - lo) <= 1e-5 * abs(lo)
    for l in range(s.L):
        _close(g[s.woff[l]:s.boff[l]], go[s.woff[l]:s.boff[l]], 2e-4)
        _close(g[s.boff[l]:s.boff[l] + s.lo[l]], go[s.boff[l]:s.boff[l] + s.lo[l]], 2e-4)
    n.close()


def test_spectral_term_gradient_matches_oracle():
    dil = (1, 2, 4)
    n = _net(4, 2, 16, dil, 2)
    s = O.Shape(4, 2, 16, dil)
    rng = np.random.default_rng(6)
    x = rng.standard_normal((3, 4, 96)).astype(np.float32)
    y = rng.standard_normal((3, 2, 96)).astype(np.float32)
    M = rng.standard_normal((64, 64))
    K = (M @ M.T / 64.0).astype(np.float32)
    n.set_spectral(K, 32, 0.8)
    p = n.params()
    loss, g = n.loss_grad(x, y, 20)
    lo, go = O.loss_and_grad(s, p.astype(np.float64), x.astype(np.float64), y.astype(np.float64),
                             20, spectral=(K.astype(np.float64), 32, 0.8))
    assert abs(loss - lo) <= 1e-4 * abs(lo), (loss, lo)
    _close(g, go, 2e-4)
    n.set_spectral(None, 0, 0.0)
    l2, _ = n.loss_grad(x, y, 20)
    l2o, _ = O.loss_and_grad(s, p.astype(np.float64), x.astype(np.float64), y.astype(np.float64), 20)
    assert abs(l2 - l2o) <= 1e-5 * abs(l2o)
    n.close()


def test_adam_step_matches_oracle():
    dil = (1, 2, 4)
    n = _net(2, 2, 16, dil, 3)
    s = O.Shape(2, 2, 16, dil)
    rng = np.random.default_rng(8)
    x = rng.standard_normal((6, 2, 64)).astype(np.float32)
    y = rng.standard_normal((6, 2, 64)).astype(np.float32)
    n.set_data(x, y)
    p = n.params()
    adam = O.Adam(s.count, 1e-3)
    # the third step clips the gradient to a tenth of its norm
    for step, (idx, clip) in enumerate((([0, 2, 4], 0.0), ([5, 1, 3], 0.0), ([1, 1, 0], -1.0))):
        lo, go = O.loss_and_grad(s, p.astype(np.float64), x[idx].astype(np.float64),
                                 y[idx].astype(np.float64), 10)
        gn = float(np.sqrt(np.sum(go ** 2)))
        if clip < 0:
            clip = 0.1 * gn
        loss = n.train_batch(idx, 10, 1e-3, clip)
        assert abs(loss - lo) <= 1e-5 * abs(lo), step
        assert abs(n.last_grad_norm - gn) <= 1e-4 * gn, (n.last_grad_norm, gn)
        p = adam.step(p, go.astype(np.float32), clip)
        _close(n.params(), p, 1e-5)
    n.close()


def test_training_reduces_the_loss():
    """A small net learns to continue damped sinusoids from their first
    quarter: the held-out loss falls by 4x in 1500 steps (the CPU oracle,
    trained the same way, reaches 6.7x)."""
    from ems_amd.learn import ConvNet
    rng = np.random.default_rng(21)
    T, N = 128, 32
    t = np.arange(T)

    def batch(n):
        f = rng.uniform(0.03, 0.08, n)[:, None]
        a = rng.uniform(0.01, 0.04, n)[:, None]
        ph = rng.uniform(0, 2 * np.pi, n)[:, None]
        y = np.exp(-a * t) * np.sin(2 * np.pi * f * t + ph)
        x = np.zeros((n, 2, T), np.float32)
        x[:, 0, :N] = y[:, :N]
        x[:, 1, :N] = 1.0
        return x, y[:, None, :].astype(np.float32)

    xs, ys = batch(512)
    xh, yh = batch(64)
    net = ConvNet(2, 1, 32, (1, 2, 4, 8, 16), seed=5)
    net.set_data(xs, ys)
    before = float(np.mean((net.forward(xh)[:, :, N:] - yh[:, :, N:]) ** 2))
    for it in range(1500):
        net.train_batch(rng.integers(0, 512, 32), N, 2e-3)
    after = float(np.mean((net.forward(xh)[:, :, N:] - yh[:, :, N:]) ** 2))
    assert after < before / 4.0, (before, after)
    net.close()


def test_invalid_arguments():
    from ems_amd.learn import ConvNet
    from ems_amd._native import EmsError
    n = ConvNet(2, 1, 8, (1, 2), seed=0)
    with pytest.raises(EmsError):
        n.forward(np.zeros((1, 3, 10), np.float32))
    with pytest.raises(EmsError):
        n.set_params(np.zeros(3, np.float32))
    n.set_data(np.zeros((4, 2, 10), np.float32), np.zeros((4, 1, 10), np.float32))
    with pytest.raises(EmsError):
        n.train_batch([0, 4], 0, 1e-3)
    n.close()


# Shapes at the edges of the convolutions' tiles: single samples and
# channels, channels past and short of 16, 32 and 64, dilations that do not
# divide the length, that exceed a block and that exceed the sequence,
# lengths around a block's 64 samples, and a batch that fills the chip (waves
# of eight output channels in training; the others one).
EDGES = [(1, 1, 1, (1, 1), 1, 1), (5, 3, 33, (3, 40), 2, 257), (4, 2, 48, (1, 2, 64, 100), 3, 130),
         (17, 18, 70, (7, 65, 200), 2, 96), (4, 2, 130, (2, 31), 1, 65), (2, 1, 32, (5, 1), 9, 63),
         (4, 2, 64, (1, 2, 4, 8, 16, 32), 5, 500), (5, 3, 52, (3, 40), 44, 257)]


@pytest.mark.parametrize("shape", EDGES)
def test_edge_shapes_match_oracle(shape):
    """Outputs and gradients against the oracle, the tolerances of the tests
    above (sums of up to 9 * 130 products in f32, in another order)."""
    cin, cout, ch, dil, B, T = shape
    n = _net(cin, cout, ch, dil, 11)
    s = O.Shape(cin, cout, ch, dil)
    rng = np.random.default_rng(T)
    p = n.params() + rng.standard_normal(s.count).astype(np.float32) * 0.02
    n.set_params(p)
    x = rng.standard_normal((B, cin, T)).astype(np.float32)
    y = rng.standard_normal((B, cout, T)).astype(np.float32)
    _close(n.forward(x), O.forward(s, p.astype(np.float64), x.astype(np.float64)), 2e-5)
    for b in (B, 1):  # (the second call in buffers sized for the first)
        loss, g = n.loss_grad(x[:b], y[:b], T // 3)
        lo, go = O.loss_and_grad(s, p.astype(np.float64), x[:b].astype(np.float64),
                                 y[:b].astype(np.float64), T // 3)
        assert abs(loss - lo) <= 1e-5 * abs(lo)
        for l in range(s.L):
            _close(g[s.woff[l]:s.boff[l]], go[s.woff[l]:s.boff[l]], 2e-4)
            _close(g[s.boff[l]:s.boff[l] + s.lo[l]], go[s.boff[l]:s.boff[l] + s.lo[l]], 2e-4)
    # more sequences than the first calls, shorter ones
    z = rng.standard_normal((4 * B + 1, cin, max(1, T // 4))).astype(np.float32)
    _close(n.forward(z), O.forward(s, p.astype(np.float64), z.astype(np.float64)), 2e-5)
    n.close()


def test_infinite_and_tiny_inputs():
    """An infinite sample saturates tanh as the plain sums do; samples at the
    bottom of f32's range do not disturb the others."""
    dil = (1, 2)
    n = _net(2, 1, 40, dil, 3)
    s = O.Shape(2, 1, 40, dil)
    p = n.params()
    x = np.random.default_rng(2).standard_normal((2, 2, 90)).astype(np.float32)
    x[0, 0, 17] = np.inf
    x[1, 1, 40:50] = np.float32(1e-42)
    got = n.forward(x)
    assert np.all(np.isfinite(got))
    _close(got, O.forward(s, p.astype(np.float64), x.astype(np.float64)), 2e-5)
    n.close()


def _free():
    """Free device memory (the runtime that the library is linked with)."""
    a, b = C.c_size_t(), C.c_size_t()
    assert nat.lib.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
    return a.value


def test_prediction_needs_no_training_memory():
    """Creating a network and predicting allocate the parameters, the
    gradient, Adam's two moments and the packed bf16 weights (18 bytes a
    parameter and the padded first and last layers); the rows that training
    reads come with the first training call."""
    cin, cout, ch, dil = 32, 32, 1024, (1, 2, 4)
    x, y = np.zeros((1, cin, 16), np.float32), np.zeros((1, cout, 16), np.float32)
    small = _net(cin, cout, 64, (1, 2), 1)  # (the runtime's own first allocations)
    small.loss_grad(x, y, 0)
    start = _free()
    n = _net(cin, cout, ch, dil, 1)
    n.forward(x)
    used = start - _free()
    assert used < 20 * n.param_count, used / n.param_count
    n.loss_grad(x, y, 0)
    assert start - _free() > used + 7 * n.param_count
    n.close()
    small.close()


def test_training_memory_of_one_long_trace():
    """A batch of one trace takes nine buffers of its length (inputs, targets,
    output, its gradient, the hidden layer's two, three of the backward pass);
    the spectral term's errors, padded to eight rows, come with that term."""
    T = 1 << 24
    n = _net(1, 1, 1, (1, 2), 1)
    x = np.zeros((1, 1, T), np.float32)
    n.loss_grad(x[:, :, :64], x[:, :, :64], 0)
    start = _free()
    n.loss_grad(x, x, 0)
    used = start - _free()
    assert used < 9.5 * 4 * T, used / (4 * T)
    n.set_spectral(np.eye(64, dtype=np.float32), 8, 0.5)
    y = np.full((1, 1, T), 1.0, np.float32)
    loss, _ = n.loss_grad(x, y, 0)
    # (without biases zeros give zeros: d = -1, d^T K d = 64)
    assert abs(loss - (1.0 + 0.5 * 64)) < 1e-4
    n.close()


def test_sequences_past_2_to_the_30():
    """A training step on two traces of more than 2^30 samples (2^31 in all)
    whose last 4096 samples alone are not zero, the loss over the last 2048:
    what a step on those 4096 gives. The sums of a weight's gradient hold the
    same terms in other partial sums (1e-4 of the norm); a learning rate of
    1e-3 moves every parameter by that much, the gradient's sign deciding."""
    tail, T = 4096, (1 << 30) + 4096
    rng = np.random.default_rng(3)
    xs = rng.standard_normal((1, 1, tail)).astype(np.float32)
    ys = rng.standard_normal((1, 1, tail)).astype(np.float32)
    got = []
    for length in (tail, T):
        n = _net(1, 1, 1, (3, 5), 1)
        x, y = np.zeros((1, 1, length), np.float32), np.zeros((1, 1, length), np.float32)
        x[:, :, -tail:], y[:, :, -tail:] = xs, ys
        n.set_data(x, y)
        del x, y
        loss = n.train_batch([0, 0], length - 2048, 1e-3)
        got.append((loss, n.last_grad_norm, n.params()))
        n.close()
    (l0, g0, p0), (l1, g1, p1) = got
    assert g0 > 0.0 and abs(l1 - l0) <= 1e-5 * l0 and abs(g1 - g0) <= 1e-4 * g0
    assert np.abs(p1 - p0).max() <= 1e-5


@pytest.mark.parametrize("shape", EDGES[:4], ids=str)
def test_weight_rows_follow_the_optimizer(shape):
    """Gradients after optimizer steps, whose weight rows the steps wrote, are
    those of the same parameters packed afresh, bit for bit."""
    cin, cout, ch, dil, B, T = shape
    n, fresh = _net(cin, cout, ch, dil, 5), _net(cin, cout, ch, dil, 6)
    rng = np.random.default_rng(T)
    x = rng.standard_normal((B, cin, T)).astype(np.float32)
    y = rng.standard_normal((B, cout, T)).astype(np.float32)
    n.set_data(x, y)
    for _ in range(3):
        n.train_batch(np.arange(B), T // 3, 1e-2)
        fresh.set_params(n.params())
        for a, b in zip(n.loss_grad(x, y, 0), fresh.loss_grad(x, y, 0)):
            assert np.array_equal(np.float32(a).view(np.uint32), np.float32(b).view(np.uint32))
    n.close()
    fresh.close()


def test_predictions_past_one_launch():
    """More sequences than the blocks of one launch hold: every one's output
    is that of its own short call."""
    B = 9_000_000
    n = _net(1, 1, 1, (1, 2), 4)
    x = np.random.default_rng(1).standard_normal((B, 1, 1)).astype(np.float32)
    got = n.forward(x)
    for at in (0, (1 << 22) - 3, (1 << 23) - 3, B - 6):
        few = n.forward(x[at:at + 6])
        assert np.array_equal(got[at:at + 6].view(np.uint32), few.view(np.uint32)), at
    n.close()
