"""The f64 adjoint's helicity sums (tp_helicity.h, helicity_gradients) with
photons that have no energy, which RAMBO makes from given points with u1 u2 = 1:
their spinors are zero, so the sums of B+ and B- are 0 and the others, whose
amplitudes the reference divides 0 by 0, no number."""
import numpy as np
import pytest

from test_helgrad import helgrad, run_constants  # noqa: F401 (fixture)
from test_helicity import helicity  # noqa: F401 (fixture)


def momenta(rest, along):
    """Photons `rest` without energy; `along`: another one exactly along -Z."""
    p = np.array([[10., 20., -5., np.sqrt(525.)], [-3., 4., 12., 13.], [8., -9., 12., 17.]])
    p[rest] = 0.
    if along is not None:
        p[along] = [0., 0., -30., 30.]
    return p


CASES = [((0,), None), ((1,), None), ((2,), None), ((0,), 2), ((2,), 1), ((0, 1), None), ((0, 2), 1), ((0, 1, 2), None)]


@pytest.mark.parametrize("rest,along", CASES)
def test_photons_without_energy(helicity, helgrad, valeurs, rest, along):  # noqa: F811
    e, g = run_constants(valeurs)
    p = np.array([momenta(list(rest), along)])
    assert np.array_equal(helicity("tp_helicity_spinors", e, p, g)[0, 1:3], [0., 0.])
    m, d = helgrad("tp_helgrad_closed", e, g, p)
    assert np.array_equal(m[0], [np.nan, 0., 0., np.nan, np.nan], equal_nan=True)
    assert np.isnan(d[0, 0]).any()


def test_a_photon_without_a_spinor_stays_no_number(helicity, helgrad, valeurs):  # noqa: F811
    """E below -Z beside a photon without energy: 0 times no number."""
    e, g = run_constants(valeurs)
    p = momenta([0], None)
    p[1] = [1., 1., -30., 29.]
    p = np.array([p])
    assert np.isnan(helicity("tp_helicity_spinors", e, p, g)).all()
    assert np.isnan(helgrad("tp_helgrad_closed", e, g, p)[0]).all()
