"""The directional kernels of the per-block path at the edges of their tiles
(needs a GPU): 63 cells along x, 16 columns by 15 cells along y and z, one
cell less and one more of each.  dq <= 1e-12 of the row's largest value
against the oracle, as for the larger blocks."""
import numpy as np
import pytest

from _util import cases, oracle_for, pkg, rel_err
import oracle as O

pytestmark = pytest.mark.gpu

CELLS = [([15], [7], [16]), ([16], [15], [7]), ([17], [31], [8]), ([7], [16], [30]), ([64], [14], [15]), ([63], [8], [14])]


@pytest.mark.parametrize("scheme,recon", [(51, 2), (71, 2), (52, 2), (72, 2), (3, 2), (2, 3), (6, 2)])
@pytest.mark.parametrize("cells", CELLS, ids=["x".join("+".join(map(str, a)) for a in c) for c in CELLS])
def test_pencil_tiles(cells, scheme, recon):
    print(f"[gpu] pencils {cells} scheme {scheme} recon {recon}", flush=True)
    case = cases.mixing_layer_case(*cells, scheme=scheme, reconstruction=recon, perturbation=2e-2)
    o = oracle_for(case)
    s = pkg.Solver(case)
    s.setup_mixing_layer()
    s.set(0, pkg.FIELD_BV, o.array(0, O.BV))
    s.initialize()
    o.rhs(0)
    s.compute_rhs(0)
    e = rel_err(s.get(0, pkg.FIELD_DQ), o.array(0, O.DQ))
    s.close()
    assert np.all(e <= 1e-12), e
