"""Transposed boundary copies of opposite faces (needs a GPU): on axes of up to
2 ngg + 1 nodes the two periodic copies read common cells, so their transposes
may not share a launch; on longer axes they do.  Gradient against the tangent
oracle as for the larger boxes."""
import numpy as np
import pytest

from _util import cases
from test_gpu_adjoint import _gpu_gradient, _tangent_gradient

pytestmark = pytest.mark.gpu


# 7 nodes: both copies read node 3.  On 6 nodes the modes' amplitudes hardly reach theta (oracle gradient 4e-13 after
# 7 steps against 6e-8 on 7 nodes), so the bound, 1e-9 of it, would lie at 1e-21, below the rounding (1e-20).
# On 9 nodes some stencils have three points that differ by rounding between two equal jumps: tau and beta_1 are then
# rounding errors, and so are the weights (one unit in the last place of the state moves the oracle's dq of rho by
# 1.5e-7 of its largest value there, by 4e-14 on 11 nodes).
@pytest.mark.parametrize("n", [7, 8, 10])
def test_gradient_on_short_axes(n):
    print(f"[gpu] adjoint gradient, {n}^3, 7 steps", flush=True)
    case = cases.fourier_case(n, n_steps=7, checkpoint_every=3)
    th_g, g = _gpu_gradient(case, 3)
    th_o, g_o = _tangent_gradient(case)
    err = np.abs(g - g_o)
    assert abs(th_g - th_o) <= 1e-12 * abs(th_o)
    assert np.all(err <= 1e-9 * np.max(np.abs(g_o)) + 1e-7 * np.abs(g_o)), (g, g_o)
