"""A NaN temperature in the mixture path (needs a GPU) reaches everything that
is formed from it at its node -- the energy, cp, gamma, the sound speed, the
transport properties -- and nothing at other nodes."""
import numpy as np
import pytest

from _util import pkg

pytestmark = pytest.mark.gpu

MX = pkg.mixture


def test_nan_temperature_is_not_replaced():
    tg = MX.load_mechanism(*MX.H2_AIR_FILES)
    case = pkg.cases.reacting_single_block(12, 16, 10, tg)
    print("[gpu] fr NaN temperature at one node", flush=True)
    s = MX.FrSolver(case, tg)
    s.setup_mixing_layer()
    bv = s.get(0, MX.FIELD_BV)
    k, j, i = 7, 9, 8  # an interior node that no ghost node copies
    bv[5, k, j, i] = np.nan
    s.set(0, MX.FIELD_BV, bv)
    s.initialize()
    for f in (MX.FIELD_CP, MX.FIELD_GAMMA, MX.FIELD_C, MX.FIELD_MUL, MX.FIELD_LAMBDA, MX.FIELD_RHOD):
        a = s.get(0, f)
        assert np.all(np.isnan(a[:, k, j, i])), f
        assert np.count_nonzero(~np.isfinite(a)) == a.shape[0], f
    cv = s.get(0, MX.FIELD_CV)
    assert np.isnan(cv[4, k, j, i]) and np.count_nonzero(~np.isfinite(cv)) == 1
    s.close()
