"""Periodic axes of the mixture path with no more nodes than ghost layers
(needs a GPU), the thinnest blocks that are accepted: a ghost layer's source by
the reference's loop is then itself a ghost node.  The ghost layers of a noisy
state after initialisation against the oracle's sequential copies, exactly;
after two steps, batched and per block, every ghost layer against the interior
node it continues, exactly."""
import numpy as np
import pytest

from _util import pkg
import mech
import oracle_fr as OF

pytestmark = pytest.mark.gpu

MX = pkg.mixture


def _continuation(m, g):
    """Padded index that each padded index of a periodic axis continues: layer l below node 0 is node m - 1 - l,
    above node m - 1 node l, both by whole periods of m - 1 cells (l = m - 1: node 0 and node m - 1)."""
    low = [m - 2 - (l - 1) % (m - 1) for l in range(g, 0, -1)]
    high = [1 + (l - 1) % (m - 1) for l in range(1, g + 1)]
    return np.array(low + list(range(m)) + high) + g


@pytest.mark.parametrize("scheme", [51, 71])
@pytest.mark.parametrize("nx,nz", [(9, 2), (9, 3), (9, 4), (2, 9), (3, 9), (4, 3)])
def test_ghost_layers_of_thin_axes(nx, nz, scheme):
    tg, to = MX.load_mechanism(*MX.H2_AIR_FILES), mech.load(*MX.H2_AIR_FILES)
    case = pkg.cases.reacting_single_block(nx, 9, nz, tg, scheme=scheme)
    print(f"[gpu] fr thin periodic axes {nx} x 9 x {nz}, scheme {scheme}", flush=True)
    o = OF.FrOracle(case, to)
    o.setup_mixing_layer()
    bv = o.array(0, OF.BV)
    rng = np.random.default_rng(5)
    g = (bv.shape[1] - nz) // 2
    noise = 1.0 + 1e-3 * rng.standard_normal(bv[:5].shape)
    bv[:5] *= noise  # rho, velocity, p; the first and the last node of an axis differ, too
    runs = []
    for mode in (MX.MODE_BATCHED, MX.MODE_DIRECT):
        s = MX.FrSolver(case, tg)
        s.setup_mixing_layer()
        s.set(0, MX.FIELD_BV, bv)
        s.initialize()
        runs.append((s, mode))
    o.initialize()
    cx, cz = _continuation(nx, g), _continuation(nz, g)
    for s, mode in runs:
        for fo, fg in ((OF.BV, MX.FIELD_BV), (OF.SV, MX.FIELD_SV)):
            np.testing.assert_array_equal(s.get(0, fg), o.array(0, fo))
        s.rk3(2, mode)
        for f in (MX.FIELD_BV, MX.FIELD_SV):
            a = s.get(0, f)
            assert np.all(np.isfinite(a)), f
            np.testing.assert_array_equal(a, a[:, cz])
            inner = a[:, g:-g, g:-g]
            np.testing.assert_array_equal(inner, inner[..., cx])
    for f in (MX.FIELD_BV, MX.FIELD_SV, MX.FIELD_CV):
        np.testing.assert_array_equal(runs[0][0].get(0, f), runs[1][0].get(0, f))
    for s, _ in runs:
        s.close()
