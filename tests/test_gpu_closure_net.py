"""The closure network's matrix-unit kernels at the edges of their tiles (16 or 32 samples a tile, one work-group
per tile up to 256 or 512 work-groups, several tiles per work-group beyond) and the step's kept-box closure term.

Tolerances, fixed before the first run: with FP32 unit round-off 6e-8, a dot product of 64 terms of random sign is
good to about 8 u, three layers and tanh to 2e-6 relative; the gradient adds the sum over samples. 1e-5 forward and
2e-5 gradient leave a factor of 5 or more."""
import numpy as np
import pytest

from laps_amd import closure
from tests import closure_np as ref
from tests.helpers import params, rel_l2, seeded_state

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    from laps_amd import runtime
    runtime.lib()
    return runtime


@pytest.mark.parametrize("n", (1, 15, 17, 31, 33, 4095, 4097, 8192, 16385, 40000))
def test_network_at_tile_edges(rt, n):
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, 28)).astype(np.float32)
    T = rng.standard_normal((n, 18)).astype(np.float32)
    P = (closure.init_params(n) + 0.05 * rng.standard_normal(rt.MLP_NPARAM)).astype(np.float32)
    assert rel_l2(rt.mlp_forward(X, P), ref.forward(X.astype(np.float64), P)[0]) < 1e-5
    G, loss = rt.mlp_grad(X, T, P)
    want, Gr = ref.loss_grad(X, T, P)
    assert rel_l2(G, Gr) < 2e-5
    assert loss == pytest.approx(want, rel=1e-5)


def test_tanh_range(rt):
    """first-layer pre-activations from 1e-6 to 30 of both signs, infinities and NaN: the network as numpy has it"""
    v = np.concatenate([np.logspace(-6, 1.5, 400), [0.0, 0.5499, 0.5501, 88.0, 1e30, np.inf]])
    v = np.concatenate([v, -v]).astype(np.float32)
    X = np.zeros((v.size + 1, 28), np.float32)
    X[: v.size, 0] = v
    X[v.size, 0] = np.nan
    P = np.zeros(rt.MLP_NPARAM, np.float32)
    P[0] = 1.0                                              # h1[0] = tanh(x0)
    P[28 * 64 + 64] = 1e-3                                  # z2[0] = h1[0] / 1000: tanh is linear there to 3e-7
    P[28 * 64 + 64 + 64 * 64 + 64] = 1e3                    # y[0] = 1000 h2[0]
    Y = rt.mlp_forward(X, P)
    with np.errstate(invalid="ignore"):
        want = ref.forward(X.astype(np.float64), P)[0][:, 0]   # an infinity times a zero weight is NaN
    assert np.array_equal(np.isnan(Y[:, 0]), np.isnan(want))
    ok = ~np.isnan(want)
    assert ok.sum() >= v.size - 2
    assert np.max(np.abs(Y[ok, 0] - want[ok]) / np.maximum(np.abs(want[ok]), 1e-30)) < 1e-6


@pytest.mark.parametrize("n,dealias", (((32, 16, 64), 1), ((96, 32, 16), 2), ((16, 96, 32), 3)))
def test_kept_box_term_of_the_step(rt, n, dealias):
    """the closure's share of one short step (dt = 1e-6: dt times its right-hand side to a few 1e-5) against the
    full-spectrum term of closure_eval, for every mask (the filter's rows are padded past nx/2 + 1)"""
    p = params(n, dealias_option=dealias, Ly=3.0)
    uu, pr = seeded_state(p, seed=3, kmax=4, du=0.2, db=0.2)
    rng = np.random.default_rng(4)
    vec = closure.closure_vector(closure.init_params(5), np.zeros(28, np.float32),
                                 (0.5 + rng.random(28)).astype(np.float32), np.full(18, 1e-2, np.float32))
    dt = 1e-6
    with rt.Laps(p) as a, rt.Laps(p) as b:
        for g in (a, b):
            g.set_state(uu, pr)
            g.set_fixed_dt(dt)
            g.step(1)           # dealiased from here on
        b.closure_set(vec)
        rhs = b.closure_eval()[1]
        a.step(1)
        b.step(1)
        d = (b.spectral() - a.spectral())[..., 1:] / dt
    kept = np.abs(d).sum(-1) > 0
    assert kept.sum() > 100
    f = np.ones(n[0] // 2 + 1)
    if dealias == 2:            # the filter multiplies the term as it does the state
        def filt(m):
            w = 2 * np.pi * m
            af = 0.495
            aj, bj, cj = (5 + 6 * af) / 8, (1 + 2 * af) / 2, -(1 - 2 * af) / 8
            return (aj + bj * np.cos(w) + cj * np.cos(2 * w)) / (1 + 2 * af * np.cos(w))
        f = (filt(np.arange(n[0] // 2 + 1) / n[0])[:, None, None] * filt(np.fft.fftfreq(n[1]))[None, :, None]
             * filt(np.fft.fftfreq(n[2]))[None, None, :])
        # three substages weigh the term by 8/15 f^3, (5/12 - 17/60) f^2 and (3/4 - 5/12) f
        f = 8 / 15 * f ** 3 + (5 / 12 - 17 / 60) * f ** 2 + (3 / 4 - 5 / 12) * f
        rhs = rhs * f[..., None]
    rhs = rhs * kept[..., None]
    assert rel_l2(d, rhs) < 1e-3
