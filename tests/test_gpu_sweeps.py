"""The row and march kernels of the batched stage at the edges of their work
lists (needs a GPU): rows shorter and longer than a wave and its 58 / 56 / 62
updated lanes, columns that leave a partial last wave, marches of one short
piece and of several, the smallest blocks, with and without viscous fluxes, and
marches of whole columns.
dq <= 1e-12 of the row's largest value against the oracle (rounding of split
fluxes that carry +-lambda rho / 2 terms, about 10^3 times dq), primitives
after two steps <= 1e-9."""
import numpy as np
import pytest

from _util import cases, interior, oracle_for, pkg, rel_err
import oracle as O

pytestmark = pytest.mark.gpu

CELLS = [([5], [5], [5]), ([57], [6], [5]), ([58], [5], [7]), ([61], [8], [9]), ([63], [9], [8]), ([130], [7], [8]),
         ([6], [70], [5]), ([8], [70], [9]), ([5], [6], [135]), ([9], [7], [135]), ([8, 59], [7], [9, 8])]


def for_z7(cells):
    """Periodic axes of at least 7 cells.  On one of 6 cells the seven points of a WENO-Z7 stencil begin and end with
    the same node.  Where the others are equal (F+ of rho where the velocity is negative and T uniform), beta_0 - beta_3
    vanishes and both inner indicators do, so the weights are those of the rounding error of beta_0 - beta_3:
    tau / (eps + beta_1)^2 up to (2^-53 beta_0 / (1e-20 beta_0))^2 = 1e8, of either sign of the error.  Any two
    orders of summation then differ (measured 1e-4 of the largest dq of rho).  There the sweeps are held to the
    per-block kernels' bits instead (test_gpu_batched_rounding.py)."""
    return [[max(n, 7) for n in axis] if d != 1 else axis for d, axis in enumerate(cells)]


# the viscous kernel does not depend on the reconstruction: without it once for each width of the stencil
@pytest.mark.parametrize("scheme,visc", [(50, 2), (51, 2), (51, 0), (71, 2), (71, 0)])
@pytest.mark.parametrize("cells", CELLS, ids=["x".join("+".join(map(str, a)) for a in c) for c in CELLS])
def test_rows_and_marches(cells, scheme, visc):
    cells = for_z7(cells) if scheme == 71 else cells
    case = cases.mixing_layer_case(*cells, scheme=scheme, viscous_order=visc, perturbation=2e-2)
    print(f"[gpu] sweeps {cells} scheme {scheme} visc {visc}", flush=True)
    o = oracle_for(case)
    s = pkg.Solver(case)
    s.setup_mixing_layer()
    for b in range(len(case["blocks"])):
        s.set(b, pkg.FIELD_BV, o.array(b, O.BV))
    s.initialize()
    for b in range(len(case["blocks"])):
        o.rhs(b)
        s.compute_rhs_batched(b)
        e = rel_err(s.get(b, pkg.FIELD_DQ), o.array(b, O.DQ))
        assert np.all(e <= 1e-12), (b, e)
    dt_o, dt_g = o.step(2), s.rk3(2, pkg.MODE_BATCHED)
    assert abs(dt_g - dt_o) <= 1e-12 * dt_o
    for b in range(len(case["blocks"])):
        e = rel_err(interior(s.get(b, pkg.FIELD_BV), s.ngg), interior(o.array(b, O.BV), s.ngg))
        assert np.all(e <= 1e-9), (b, e)
    s.close()


@pytest.mark.parametrize("scheme", [50, 51, 71])
@pytest.mark.parametrize("my,mz", [(5, 6), (7, 11), (12, 13), (64, 65)])
def test_long_marches(my, mz, scheme):
    """Blocks of so many columns that a march takes whole columns (65 nodes: two pieces): lengths around the turn of
    the unrolled march (6) and at the cut (64), where smaller blocks have marches of at most 4 cells.  Without
    viscous fluxes the per-block kernels give the same bits but for the odd root (test_gpu_batched_rounding.py)."""
    my = max(my, 6) if scheme == 71 else my  # ngg + 2 nodes at least
    mx = 262144 // my + 37  # 4096 waves along z and more along y: 16 a CU
    case = cases.mixing_layer_case([mx - 1], [my - 1], [mz - 1], scheme=scheme, viscous_order=0, perturbation=2e-2)
    print(f"[gpu] long marches {mx} x {my} x {mz} scheme {scheme}", flush=True)
    s = pkg.Solver(case)
    s.setup_mixing_layer()
    s.initialize()
    s.compute_rhs(0)
    want = s.get(0, pkg.FIELD_DQ)
    s.compute_rhs_batched(0)
    got = s.get(0, pkg.FIELD_DQ)
    s.close()
    assert np.all(np.isfinite(want)) and np.all(np.max(np.abs(want), axis=(1, 2, 3)) > 0)
    assert np.all(np.mean(got != want, axis=(1, 2, 3)) <= 1e-3)
    if my >= 7:  # short periodic axes: for_z7
        assert np.all(rel_err(got, want) <= 1e-12)
