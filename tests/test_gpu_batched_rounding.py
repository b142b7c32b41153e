"""The sweeps and the update of a batched stage round as the per-block kernels
do (needs a GPU): same split fluxes, faces, sums and update in the same order, so
without viscous fluxes the residual and a step's state agree bit for bit but
for the odd root (the short square root is within one unit in the last place,
not always the nearest): at most 1 in 1000 values may differ.  Products by
rounded reciprocals in place of the quotients, or fused sums, change more than
half of them."""
import numpy as np
import pytest

from _util import cases, pkg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme", [50, 51, 71])
@pytest.mark.parametrize("cells", [([33], [29], [31]), ([7, 9], [10], [8, 12]), ([6], [5], [6]),
                                   ([5], [6], [135])], ids=["one", "four", "six", "long"])
def test_inviscid_step_has_the_per_block_bits(cells, scheme):
    case = cases.mixing_layer_case(*cells, scheme=scheme, viscous_order=0, perturbation=2e-2)
    print(f"[gpu] batched rounding {cells} scheme {scheme}", flush=True)
    a, b = pkg.Solver(case), pkg.Solver(case)
    for s in (a, b):
        s.setup_mixing_layer()
        s.initialize()
    for blk in range(len(case["blocks"])):
        a.compute_rhs(blk)
        b.compute_rhs_batched(blk)
    dq = [[s.get(blk, pkg.FIELD_DQ) for blk in range(len(case["blocks"]))] for s in (a, b)]
    a.rk3(1, pkg.MODE_PLAIN)
    b.rk3(1, pkg.MODE_BATCHED)
    for blk in range(len(case["blocks"])):
        for what, x, y in (("dq", dq[0][blk], dq[1][blk]), ("cv", a.get(blk, pkg.FIELD_CV), b.get(blk, pkg.FIELD_CV)),
                           ("bv", a.get(blk, pkg.FIELD_BV), b.get(blk, pkg.FIELD_BV))):
            differ = np.mean(x != y, axis=(1, 2, 3))
            assert np.all(differ <= 1e-3), (blk, what, differ)
    a.close()
    b.close()
