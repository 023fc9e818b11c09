"""Rounding of the closure network's kernels, to the last bits."""
import numpy as np
import pytest

from laps_amd import closure
from tests.helpers import params

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    from laps_amd import runtime
    runtime.lib()
    return runtime


@pytest.mark.parametrize("lo,hi", ((1e-4, 0.5), (0.5, 0.6), (0.6, 0.7), (0.7, 1.0), (1.0, 1.1), (1.1, 12.0)))
def test_tanh_within_the_library(rt, lo, hi):
    """A network that hands tanh(x) through: the second layer's input is 2^-20 tanh(x), where tanh is the identity to
    3e-13, and the third multiplies by 2^20; every other product is exact or zero. The error against FP64 stays
    below 1.5 units in the last place of the result; the device library's tanhf has 1.405 at most over all floats."""
    a, b = (int(np.float32(v).view(np.uint32)) for v in (lo, hi))
    x = np.unique(np.linspace(a, b, 400_000).astype(np.uint32)).view(np.float32)
    x[1::2] *= -1
    X = np.zeros((x.size, 28), np.float32)
    X[:, 0] = x
    P = np.zeros(rt.MLP_NPARAM, np.float32)
    P[0] = 1.0
    P[28 * 64 + 64] = 2.0 ** -20
    P[28 * 64 + 64 + 64 * 64 + 64] = 2.0 ** 20
    y = rt.mlp_forward(X, P)[:, 0].astype(np.float64)
    want = np.tanh(x.astype(np.float64))
    ulp = 2.0 ** (np.frexp(want)[1] - 24)
    assert np.max(np.abs(y - want) / ulp) < 1.5


@pytest.mark.parametrize("n", (1, 33, 4096, 4097, 16385, 100_000, 262_145))
def test_loss_is_summed_in_fp64(rt, n):
    """The mean squared error of a batch against an FP64 sum of the FP32 squares, whose differences use the network's own
    outputs (the forward pass and the gradient share its arithmetic, row by row): one rounding to FP32, and 1e-10
    for the order of the FP64 sums. The loss of a training step is the same number."""
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, 28)).astype(np.float32)
    T = rng.standard_normal((n, 18)).astype(np.float32)
    P = (rng.standard_normal(rt.MLP_NPARAM) / 8).astype(np.float32)
    d = rt.mlp_forward(X, P) - T
    want = (d * d).astype(np.float64).sum() / (n * 18)
    half = 0.5 * np.spacing(np.float32(want))
    loss = rt.mlp_grad(X, T, P)[1]
    assert abs(float(loss) - want) <= half + 1e-10 * want
    assert np.float32(rt.mlp_train(X, T, P, 1, n, 1e-3)[1][0]) == np.float32(loss)


def test_step_features_are_quotients(rt):
    """The network of a step against the network on the handed-over features, bit for bit, where the last bit of the FP64
    gradients decides their FP32 rounding: f(x + dx) - f(x - dx) is 2 dx times a midpoint of two floats, exactly, and
    with 2 dx = 123/64 the product with the rounded reciprocal misses half of these midpoints."""
    n = (16, 32, 16)
    p = params(n, Lx=123 / 8)
    k = 2.0 - (2 * np.arange(n[1] * n[2] * 7) + 1) * 2.0 ** -24
    a = k * (2 * p.Lx / n[0])
    assert np.array_equal(a / (2 * p.Lx / n[0]), k)
    a = a.reshape(7, n[1], n[2])
    saw = np.array([0, 0.5, 0, -0.5] * (n[0] // 4))                  # differences of +-1 at every other point
    f = 4.0 * np.ones(n + (7,), order="F")                           # rho, u, B
    for q in range(1, 7):
        f[..., q] = saw[:, None, None] * a[q]
    uu, pr = np.ones(n + (8,), order="F"), np.ones(n + (4,), order="F")
    uu[..., 0] = f[..., 0]
    uu[..., 1:4] = f[..., :1] * f[..., 1:4]
    uu[..., 4:7] = f[..., 4:7]
    uu[..., 7] = 40.0
    pr[..., :3] = f[..., 1:4]
    rng = np.random.default_rng(1)
    std = np.ones(28, np.float32)
    vec = closure.closure_vector(closure.init_params(2) + 0.1 * rng.standard_normal(rt.MLP_NPARAM).astype(np.float32),
                                 np.zeros(28, np.float32), std, np.ones(18, np.float32))
    with rt.Laps(p) as g:
        g.set_state(uu, pr)
        X = g.closure_features()
        d = (f - np.roll(f, 2, 0)) / (2 * p.Lx / n[0])               # the gradient at the point one to the left
        want = np.roll(d, -1, 0).astype(np.float32)
        assert np.array_equal(X[:, 7::3], want.reshape(-1, 7, order="F"))
        g.closure_set(vec)
        Y = g.closure_eval()[0]
    assert np.array_equal(Y, rt.mlp_forward(X, vec[:rt.MLP_NPARAM]))
