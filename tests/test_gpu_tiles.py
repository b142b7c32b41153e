"""The launch configurations of the characteristic schemes' tile kernels (needs
a GPU): every tile shape with one workgroup per tile and with a persistent
grid, a stage in one kernel and split into two.  Steps <= 1e-9 against the
oracle's sequential steps; a persistent grid does the same arithmetic as one
workgroup per tile, bit for bit.  The residual of every shape is in
test_gpu_air_schemes.py.  For the component-wise schemes, whose kernels have no
tile, the configuration is kept and reported, the results do not depend on it,
and the autotuner leaves it alone."""
import numpy as np
import pytest

from _util import O, cases, interior, oracle_for, pkg, rel_err

pytestmark = pytest.mark.gpu

N_STEPS = 3


def _case(scheme):
    # more tiles of every shape than the chip has CUs, so that a grid of one workgroup a CU goes round
    case = cases.mixing_layer_case([44, 31], [50], [52], scheme=scheme)
    for tx, ty, tz in pkg.tile_shapes():
        assert sum(-(-b["mx"] // tx) * -(-b["my"] // ty) * -(-b["mz"] // tz) for b in case["blocks"]) > 256
    return case


_ORACLE = {}


def _oracle(scheme):
    if scheme not in _ORACLE:
        o = oracle_for(_case(scheme))
        _ORACLE[scheme] = (o, o.step(N_STEPS))
    return _ORACLE[scheme]


def _steps(case, *tile):
    s = pkg.Solver(case)
    s.setup_mixing_layer()
    s.initialize()
    if tile:
        s.set_tile(*tile)
    dt = s.rk3(N_STEPS, pkg.MODE_BATCHED)
    bv = [s.get(b, pkg.FIELD_BV) for b in range(len(case["blocks"]))]
    g = s.ngg
    s.close()
    return dt, bv, g


@pytest.mark.parametrize("split", [0, 1], ids=["one-kernel", "split-stage"])
@pytest.mark.parametrize("scheme", [52, 72])
@pytest.mark.parametrize("index", range(6))
def test_launch_configs_match_oracle(index, scheme, split):
    case = _case(scheme)
    print(f"[gpu] tile entry {index}, scheme {scheme}, split {split}: one workgroup per tile, one a CU", flush=True)
    o, dt_o = _oracle(scheme)
    dt, bv, g = _steps(case, index, 0, split)
    assert abs(dt - dt_o) <= 1e-12 * dt_o
    for b in range(len(case["blocks"])):
        e = rel_err(interior(bv[b], g), interior(o.array(b, O.BV), g))
        assert np.all(e <= 1e-9), (b, e)
    dt2, bv2, _ = _steps(case, index, 1, split)
    assert dt2 == dt
    for x, y in zip(bv, bv2):
        np.testing.assert_array_equal(x, y)


def test_the_sweeps_have_no_tile():
    case = cases.small_multiblock_case()
    print("[gpu] tile configuration of scheme 51", flush=True)
    _, want, _ = _steps(case)
    _, got, _ = _steps(case, 4, 2, 1)
    for x, y in zip(want, got):
        np.testing.assert_array_equal(x, y)


def test_autotune_leaves_the_sweeps_configuration_alone():
    print("[gpu] autotune of scheme 51", flush=True)
    s = pkg.Solver(cases.small_multiblock_case())
    s.setup_mixing_layer()
    s.initialize()
    for config in ((4, 2, 1), (1, 0, 0), (3, 4, 0)):
        s.set_tile(*config)
        index, ms = s.autotune(2)
        assert index == config[0] and 0 < ms < 1e3
        assert s.tile_config() == config
    s.close()


def test_autotune_of_a_characteristic_scheme():
    print("[gpu] autotune of scheme 52", flush=True)
    s = pkg.Solver(cases.small_multiblock_case(scheme=52))
    s.setup_mixing_layer()
    s.initialize()
    index, ms = s.autotune(2)
    assert 0 <= index < 6 and 0 < ms < 1e3
    assert s.tile_config()[0] == index
    s.close()
