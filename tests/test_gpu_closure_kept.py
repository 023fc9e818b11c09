"""The closure's right-hand side on the kept box, for every mask, on the set of modes that the mask's definition gives
(not on the modes that the step happens to change)."""
import numpy as np
import pytest

from laps_amd import closure
from tests.helpers import params, rel_l2, seeded_state

pytestmark = pytest.mark.gpu


def _filter(m):
    w, af = 2 * np.pi * m, 0.495
    return ((5 + 6 * af) / 8 + (1 + 2 * af) / 2 * np.cos(w) - (1 - 2 * af) / 8 * np.cos(2 * w)) / (1 + 2 * af * np.cos(w))


def _weights(n, dealias):
    """what is left of a constant term in each mode after a step of dt = 1: the mask, or with the filter f the sum of the
    three substages' weights 8/15 f^3, (5/12 - 17/60) f^2 and (3/4 - 5/12) f"""
    m = [np.arange(n[0] // 2 + 1)] + [np.rint(np.fft.fftfreq(k) * k) for k in n[1:]]
    m = np.meshgrid(*m, indexing="ij")
    if dealias == 1:
        return (9 * sum((a * (np.prod(n) // k)) ** 2 for a, k in zip(m, n)) <= np.prod(n, dtype=np.int64) ** 2).astype(float)
    if dealias == 3:
        return (9 * sum((a * (np.prod(n) // k)) ** 2 for a, k in zip(m, n)) < 2 * np.prod(n, dtype=np.int64) ** 2).astype(float)
    f = _filter(m[0] / n[0]) * _filter(m[1] / n[1]) * _filter(m[2] / n[2])
    f[np.abs(f) < 1e-12] = 0.0                  # the Nyquist planes
    return 8 / 15 * f ** 3 + (5 / 12 - 17 / 60) * f ** 2 + (3 / 4 - 5 / 12) * f


@pytest.mark.parametrize("n,dealias", (((32, 16, 64), 1), ((96, 32, 16), 2), ((16, 96, 32), 3), ((64, 32, 32), 3)))
def test_closure_term_on_the_kept_modes(n, dealias):
    """dt = 1e-6: the share of the closure in one step, divided by dt, is its right-hand side to dt times the fastest rate
    of the kept modes, a few 1e-5 of the whole. The network's outputs switch sign with the state (features divided by
    0.05), so every plane of modes holds at least a thousandth of that: 3e-2 of a plane, 0.1 asked, and 1 where a plane
    is dropped or shifted. Outside the mask nothing changes; the filter leaves 1e-12 there."""
    from laps_amd import runtime as rt
    p = params(n, dealias_option=dealias, Ly=3.0)
    uu, pr = seeded_state(p, seed=3, kmax=4, du=0.2, db=0.2)
    vec = closure.closure_vector(closure.init_params(5), np.zeros(28, np.float32), np.full(28, 0.05, np.float32),
                                 np.full(18, 1e-2, np.float32))
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
    w = _weights(n, dealias)
    kept = w != 0.0
    want = rhs * w[..., None]
    assert rel_l2(d[kept], want[kept]) < 1e-3
    if dealias != 2:
        assert not d[~kept].any()
    else:
        assert np.abs(d[~kept]).max() < 1e-9 * np.abs(d).max()
    for axis in range(3):
        for i in range(d.shape[axis]):
            s = np.take(want, i, axis)
            if s.any():
                assert rel_l2(np.take(d * kept[..., None], i, axis), s) < 0.1, (axis, i)
