"""The grouped ghost-layer launches of the batched finite-rate step (needs a
GPU): every face type in one run, the smallest blocks beside faces of several
workgroups (a partial last one), farfield and other faces in the same round,
inner faces whose edges conflict.  Against the oracle's sequential faces,
primitives and mass fractions <= 1e-9 after two steps (the bound of the
temperature iteration's stop, as in the other step tests), and the per-block
launches of the same ops bit for bit.

Periodic axes have at least 5 cells: on 4, the five points of a WENO-Z5 stencil
begin and end with the same node, beta_0 - beta_2 is a rounding error wherever
the three others agree, and the weights, tau / (eps + beta_1)^2 up to
(2^-53 / 1e-20)^2 = 1e8, are that error's (measured 2e-5 of w between two orders
of summation)."""
import numpy as np
import pytest

from _util import pkg, rel_err
import mech
import oracle_fr as OF

pytestmark = pytest.mark.gpu

MX = pkg.mixture


@pytest.mark.parametrize("cells,y_bc,spatial", [(([4, 5], [4], [4, 6]), 4, False), (([4], [5, 4], [5]), 6, True),
                                                (([20, 4], [5, 17], [4, 5]), 4, True)],
                         ids=["farfield-temporal", "outflow-spatial", "farfield-spatial"])
def test_ghost_rounds_and_levels(cells, y_bc, spatial):
    tg, to = MX.load_mechanism(*MX.H2_AIR_FILES), mech.load(*MX.H2_AIR_FILES)
    case = pkg.cases.reacting_case(*cells, tg, scheme=51, y_bc=y_bc, spatial=spatial)
    print(f"[gpu] fr ghost rounds {cells} y_bc {y_bc} spatial {spatial}", flush=True)
    o = OF.FrOracle(case, to)
    o.setup_mixing_layer()
    o.initialize()
    runs = []
    for mode in (MX.MODE_BATCHED, MX.MODE_DIRECT):
        s = MX.FrSolver(case, tg)
        s.setup_mixing_layer()
        s.initialize()
        s.rk3(2, mode)
        runs.append(s)
    o.step(2)
    g = runs[0].ngg
    for b in range(len(case["blocks"])):
        for f in (MX.FIELD_BV, MX.FIELD_SV, MX.FIELD_CV):
            np.testing.assert_array_equal(runs[0].get(b, f), runs[1].get(b, f))
        for fo, fg in ((OF.BV, MX.FIELD_BV), (OF.SV, MX.FIELD_SV)):
            e = rel_err(runs[0].get(b, fg)[:, g:-g, g:-g, g:-g], o.array(b, fo)[:, g:-g, g:-g, g:-g])
            assert np.all(e <= 1e-9), (b, fo, e)
    for s in runs:
        s.close()
