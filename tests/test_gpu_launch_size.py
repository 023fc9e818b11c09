"""Rules that go by the size of a launch: a box of a batched ensemble group, whose launches cover all boxes of the
group, against the same box on its own, bit for bit. The y forward pass takes its large form in the group and
the split form in the single box; rows of the larger launches are stored to the end of their last 64-byte piece
(full rows, whose padding lies past the Nyquist column, and masked rows), where no pass reads them."""
import numpy as np
import pytest

from laps_amd.params import LAPS_MIXED
from tests.helpers import params, seeded_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,count,kw", (
    ((64, 64, 64), 20, dict(dealias_option=2)),
    ((64, 64, 32), 56, dict(dealias_option=0, cfl=0.2, precision=LAPS_MIXED)),
    ((96, 64, 32), 24, dict(dealias_option=1, if_hall=1, ion_inertial_length=0.05)),
    ((128, 32, 64), 32, dict(dealias_option=1, precision=LAPS_MIXED, if_aeb=1, radius0=1.0, Ur0=0.5)),
    ((64, 32, 96), 12, dict(dealias_option=3, cfl=0.2, if_hall=1, ion_inertial_length=0.05)),
    ((32, 64, 64), 40, dict(dealias_option=3, cfl=0.2, precision=LAPS_MIXED))))
def test_large_launch_equals_small(n, count, kw, monkeypatch):
    from laps_amd import runtime
    monkeypatch.setenv("LAPS_FFT_PLAN", "0")
    p = params(n, **kw)
    uu, pr = seeded_state(p, seed=sum(n), kmax=6, du=0.2, db=0.2)
    e = runtime.Ensemble([p] * count)
    for i in range(count):
        e.box(i).set_state(uu, pr)
    e.step(3)
    with runtime.Laps(p) as g:
        g.set_state(uu, pr)
        g.step(3)
        want = g.spectral()
        assert np.isfinite(want).all()
        for i in (0, count // 2, count - 1):
            assert np.array_equal(e.box(i).spectral(), want)
    e.close()
