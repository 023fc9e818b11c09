"""The y forward pass in its two forms, the large one (a batched group of boxes) and the split one (the box on its own,
below 2^18 points a field), bit for bit at every length of the y axis and for every mask: each output must round alike
in both, whatever the compiler makes of the code around it."""
import numpy as np
import pytest

from laps_amd.params import LAPS_FP64, LAPS_MIXED
from tests.helpers import params, seeded_state

pytestmark = pytest.mark.gpu

CASES = [((16, ny, 16 if ny > 128 else 32), dealias, {}) for ny in (16, 32, 64, 96, 128, 256, 512) for dealias in (1, 2)]
CASES += [((16, 96, 32), dealias, {}) for dealias in (0, 3)]
CASES += [((32, 96, 16), 1, dict(if_aeb=1, if_corotating=1, radius0=1.0, Ur0=0.5, corotating_angle=0.25))]


@pytest.mark.parametrize("precision", (LAPS_FP64, LAPS_MIXED))
@pytest.mark.parametrize("n,dealias,kw", CASES)
def test_split_and_large_form(n, dealias, kw, precision, monkeypatch):
    from laps_amd import runtime
    monkeypatch.setenv("LAPS_FFT_PLAN", "0")
    p = params(n, dealias_option=dealias, cfl=0.2, precision=precision, **kw)
    uu, pr = seeded_state(p, seed=sum(n), kmax=4, du=0.2, db=0.2)
    # the group's points per field, at least a fifth of the grid kept along x: above the 2^18 of the split form
    count = 2 ** 18 * 5 // (n[0] * n[1] * n[2]) + 1
    e = runtime.Ensemble([p] * count)
    for i in range(count):
        e.box(i).set_state(uu, pr)
    e.step(3)
    with runtime.Laps(p) as g:
        g.set_state(uu, pr)
        g.step(3)
        want = g.spectral()
    assert np.isfinite(want).all()
    for i in (0, count - 1):
        assert np.array_equal(e.box(i).spectral(), want)
    e.close()
