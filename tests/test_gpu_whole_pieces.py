"""Rows of a kept box whose width is a multiple of the 64-byte piece (8 and 16 columns: 16 and 32 points with phase
shift), where the number of stored columns does not tell whether rows are cut at the mask or stored to the end of
the piece it ends in: boxes of a batched group large enough for whole pieces against the box on its own, which is not,
bit for bit (the columns past the mask reach no kept mode)."""
import numpy as np
import pytest

from laps_amd.params import LAPS_MIXED
from tests.helpers import params, seeded_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,count,kw", (
    ((16, 64, 64), 26, dict()),
    ((16, 96, 64), 34, dict(precision=LAPS_MIXED)),
    ((32, 64, 32), 26, dict(if_hall=1, ion_inertial_length=0.05))))
def test_whole_pieces_equal_cut_rows(n, count, kw, monkeypatch):
    from laps_amd import runtime
    monkeypatch.setenv("LAPS_FFT_PLAN", "0")
    p = params(n, dealias_option=3, cfl=0.2, **kw)
    uu, pr = seeded_state(p, seed=sum(n), kmax=4, du=0.2, db=0.2)
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
