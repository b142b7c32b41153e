"""A block of more nodes along z than two workgroups' worth of 65535 (needs a
GPU): the point kernels' launches must stay within the grid's limits.  A layer
that does not vary along z, on 131073 nodes and on 9 of the same spacing: the
state after initialisation and one batched step agree at every z.  The metric
is formed from node coordinates, up to 131072 spacings large, so its rounding is
2^-53 * 131072 of a spacing: bound 1e-10 of a variable's largest value."""
import numpy as np
import pytest

from _util import cases, interior, pkg

pytestmark = pytest.mark.gpu


def _run(nz):
    case = cases.mixing_layer_case([5], [6], [nz], perturbation=0.0, lz_over_delta=20.0 * nz / 8)
    s = pkg.Solver(case)
    s.setup_mixing_layer()
    s.initialize()
    start = [interior(s.get(0, f), s.ngg) for f in (pkg.FIELD_CV, pkg.FIELD_MUL)]
    s.rk3(1, pkg.MODE_BATCHED)
    end = interior(s.get(0, pkg.FIELD_BV), s.ngg)
    s.close()
    return start, end


def test_131073_nodes_along_z():
    print("[gpu] 6 x 7 x 131073 nodes", flush=True)
    (cv, mul), bv = _run(131072)
    (cv9, mul9), bv9 = _run(8)
    for a, ref in ((cv, cv9), (mul, mul9), (bv, bv9)):
        scale = np.max(np.abs(ref), axis=(1, 2, 3), keepdims=True)
        scale = np.where(scale < 1e-6 * np.max(scale), np.max(scale), scale)  # w is zero but for rounding
        assert np.all(np.abs(a - ref[:, 4:5]) <= 1e-10 * scale)
