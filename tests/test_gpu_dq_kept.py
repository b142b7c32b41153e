"""Batched steps leave a block's dq array alone (needs a GPU): what a residual
call put there is there after steps and after a reverse-mode forward run,
whichever kernels the scheme takes, with and without viscous fluxes and on
several blocks."""
import numpy as np
import pytest

from _util import cases, pkg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("visc", [2, 0])
@pytest.mark.parametrize("scheme", [50, 51, 71, 52])
def test_steps_keep_dq(scheme, visc):
    case = cases.mixing_layer_case([9, 12], [10], [8], scheme=scheme, viscous_order=visc)
    print(f"[gpu] dq over batched steps, scheme {scheme} visc {visc}", flush=True)
    s = pkg.Solver(case)
    s.setup_mixing_layer()
    s.initialize()
    before = []
    for b in range(len(case["blocks"])):
        s.compute_rhs(b)
        before.append(s.get(b, pkg.FIELD_DQ))
    s.rk3(2, pkg.MODE_BATCHED)
    for b, dq in enumerate(before):
        assert np.any(dq != 0)
        np.testing.assert_array_equal(s.get(b, pkg.FIELD_DQ), dq)
    s.close()


def test_adjoint_forward_keeps_dq():
    case = cases.fourier_case(10, n_steps=3, checkpoint_every=2)
    print("[gpu] dq over a reverse-mode forward run", flush=True)
    s = pkg.Solver(case)
    s.setup_fourier_case()
    s.compute_rhs(0)
    dq = s.get(0, pkg.FIELD_DQ)
    s.adjoint_forward(3, 2, case["theta"])
    np.testing.assert_array_equal(s.get(0, pkg.FIELD_DQ), dq)
    s.close()
