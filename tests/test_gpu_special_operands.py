"""Zero and infinite operands of the short reciprocal, quotient and root
sequences (needs a GPU) give what IEEE divisions and roots give.  Air: a node
with T = 0 or with a zero metric row splits its fluxes with lambda = |U| (the
per-block kernels call sqrt; dq <= 1e-12 of the row's largest value, as between
these paths elsewhere).  Mixture: rho_D, proportional to 1 / p, is infinite at
p = 0 and zero at an infinite p."""
import numpy as np
import pytest

from _util import cases, pkg, rel_err

pytestmark = pytest.mark.gpu

MX = pkg.mixture
NODE = (7, 8, 9)  # k, j, i of the padded block, interior


@pytest.mark.parametrize("scheme", [50, 51, 71])
@pytest.mark.parametrize("what", ["T", "metric"])
def test_split_fluxes_of_a_zero_wave_speed(what, scheme):
    case = cases.mixing_layer_case([12], [12], [12], scheme=scheme, perturbation=2e-2)
    print(f"[gpu] zero {what} at one node, scheme {scheme}", flush=True)
    s = pkg.Solver(case)
    s.setup_mixing_layer()
    s.initialize()
    k, j, i = NODE
    if what == "T":
        bv = s.get(0, pkg.FIELD_BV)
        bv[5, k, j, i] = 0.0
        s.set(0, pkg.FIELD_BV, bv)
    else:
        met = s.get(0, pkg.FIELD_METRIC)
        met[:, k, j, i] = 0.0
        s.set_geometry(0, s.get(0, pkg.FIELD_JAC), met)
    s.compute_rhs(0)
    want = s.get(0, pkg.FIELD_DQ)
    s.compute_rhs_batched(0)
    got = s.get(0, pkg.FIELD_DQ)
    s.close()
    assert np.all(np.isfinite(want))
    e = rel_err(got, want)
    assert np.all(e <= 1e-12), e


def test_diffusivity_of_a_zero_and_an_infinite_pressure():
    tg = MX.load_mechanism(*MX.H2_AIR_FILES)
    case = pkg.cases.reacting_single_block(12, 16, 10, tg)
    print("[gpu] fr zero and infinite pressure at one node each", flush=True)
    s = MX.FrSolver(case, tg)
    s.setup_mixing_layer()
    bv = s.get(0, MX.FIELD_BV)
    bv[4][6, 8, 7] = 0.0
    bv[4][8, 8, 7] = np.inf
    s.set(0, MX.FIELD_BV, bv)
    s.initialize()
    rd = s.get(0, MX.FIELD_RHOD)
    s.close()
    assert np.all(rd[:, 6, 8, 7] == np.inf), rd[:, 6, 8, 7]
    assert np.all(rd[:, 8, 8, 7] == 0.0), rd[:, 8, 8, 7]
