"""The mass equation taken from the momentum spectrum (no transform of the mass flux) and the induction equation
formed in the z pass, against the oracle's transformed fluxes: white-noise states, whose modes fill the spectrum
past every mask and on the Nyquist planes, on non-cubic grids, for every dealiasing option, precision and box.

Tolerance: the oracle parity bar of the double-precision step, 1e-11; for mixed precision FP32 transforms over
three steps, 1e-5."""
import numpy as np
import pytest

from laps_amd.ic import cons_from_prim
from tests.helpers import params, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", ((0, 1e-11), (1, 1e-5)))
@pytest.mark.parametrize("n,dealias,hall,aeb", (
    ((16, 32, 64), 0, 0, 0), ((32, 16, 16), 0, 1, 1), ((32, 64, 16), 1, 1, 0), ((96, 16, 32), 1, 0, 1),
    ((16, 96, 32), 2, 1, 0), ((64, 16, 96), 2, 1, 1), ((32, 32, 96), 3, 1, 1), ((64, 32, 16), 3, 0, 0)))
def test_white_noise_state_vs_oracle(oracle_mod, n, dealias, hall, aeb, precision, tol):
    from laps_amd.runtime import Laps
    kw = dict(dealias_option=dealias, cfl=0.1, viscosity=0.02, resistivity=0.02)
    if hall:
        kw.update(if_hall=1, ion_inertial_length=0.02)
    if aeb:
        kw.update(if_aeb=1, if_corotating=1, radius0=1.0, Ur0=0.5, corotating_angle=0.3)
    p = params(n, **kw)
    rng = np.random.default_rng(sum(n) + dealias)
    prim = np.zeros(n + (8,), order="F")
    prim[..., 0] = 1.0 + 0.05 * rng.standard_normal(n)
    prim[..., 1:7] = 0.05 * rng.standard_normal(n + (6,))
    prim[..., 4] += 1.0
    prim[..., 7] = 1.0 + 0.05 * rng.standard_normal(n)
    uu, pr = cons_from_prim(prim, p.adiabatic_index)
    o = oracle_mod.Oracle(p)
    o.set_state(uu, pr)
    p.precision = precision
    with Laps(p) as g:
        g.set_state(uu, pr)
        for dt in (2e-3, 2e-3, 1e-3):
            g.set_fixed_dt(dt)
            o.set_fixed_dt(dt)
            g.step(1)
            o.step(1)
        got, want = g.spectral(), o.spectral()
    o.close()
    for v in range(8):
        assert rel_l2(got[..., v], want[..., v]) < tol, v
