"""The chemical source term's distance from extended precision (needs a GPU).

Its exponents (b log T - Ea / T, up to 170, and the reaction's change of Gibbs
energy) turn a rounding of 2^-53 into 2e-14 of a rate, so comparisons in 64 bits
share the reference's rounding of Ea / T and cannot tell which side is closer.
Here the residual of uniform states at rest (unit metric: the fluxes cancel
exactly and dq is the source) is compared with the reference's formulas
(src/FiniteRateChem.cu:7-195) in extended precision: relative to the species'
gross rate (creation + destruction), root mean square over the states, no
further off than the same formulas in 64-bit numpy, whose error is printed
beside it."""
import numpy as np
import pytest

from _util import pkg

pytestmark = pytest.mark.gpu

MX = pkg.mixture
RU, PATM = 8314.462618, 101325.0


def _rates(T, rho, t, Y, real):
    """(net, gross) mass rates of every species, [n_spec][state], in the number type `real`, the quotients, powers
    and exponentials as the reference writes them."""
    ns, R = T.n_spec, real
    rho, t, Y = rho.astype(R), t.astype(R), Y.astype(R)
    c = [rho * Y[l] / R(T.mw[l]) * R(1e-3) for l in range(ns)]
    g = []
    for l in range(ns):
        tt = np.maximum(t, R(T.t_low[l]))
        a = [np.where(tt < R(T.t_mid[l]), R(T.low_coeff[l][k]), R(T.high_coeff[l][k])) for k in range(7)]
        g.append(a[0] * (R(1) - np.log(tt)) - R(0.5) * a[1] * tt - a[2] * tt ** 2 / R(6) - a[3] * tt ** 3 / R(12) -
                 R(0.05) * a[4] * tt ** 4 + a[5] / tt - a[6])
    made, lost = [np.zeros_like(t) for _ in range(ns)], [np.zeros_like(t) for _ in range(ns)]
    use_kc = any(T.label[i] != 0 and T.rev_type[i] != 1 for i in range(T.n_reac))

    def k(A, b, E):
        return R(A) * t ** R(b) * np.exp(-R(E) / t)

    for i in range(T.n_reac):
        ty = T.label[i]
        kf = k(T.A[i], T.b[i], T.Ea[i])
        cc = sum(c[l] * R(T.third_body_coeff[i][l]) for l in range(ns))
        if ty == 3:
            kf = kf + k(T.A2[i], T.b2[i], T.Ea2[i])
        elif ty == 4:
            kf = kf * cc
        elif ty > 4:
            pr = k(T.A2[i], T.b2[i], T.Ea2[i]) * cc / kf
            F = R(1)
            if ty > 5:
                al = R(T.troe_alpha[i])
                fc = (R(1) - al) * np.exp(-t / R(T.troe_t3[i])) + al * np.exp(-t / R(T.troe_t1[i]))
                if ty == 7:
                    fc = fc + np.exp(-R(T.troe_t2[i]) / t)
                lf, lp = np.log10(fc), np.log10(pr)
                q = lp - R(0.4) - R(0.67) * lf
                F = R(10) ** (lf / (R(1) + (q / (R(0.75) - R(1.27) * lf - R(0.14) * q)) ** 2))
            kf = kf * pr / (R(1) + pr) * F
        kb = np.zeros_like(t)
        if ty != 0:
            assert use_kc and T.rev_type[i] != 1  # all this mechanism has
            dg = sum(g[l] * R(T.stoi_b[i][l] - T.stoi_f[i][l]) for l in range(ns))
            kb = kf / ((R(PATM) / R(RU) * R(1e-3) / t) ** T.order[i] * np.exp(-dg))
        for l in range(ns):
            kf = kf * c[l] ** T.stoi_f[i][l] if T.stoi_f[i][l] else kf
            kb = kb * c[l] ** T.stoi_b[i][l] if ty != 0 and T.stoi_b[i][l] else kb
        for l in range(ns):
            made[l] = made[l] + kb * R(T.stoi_f[i][l]) + kf * R(T.stoi_b[i][l])
            lost[l] = lost[l] + kf * R(T.stoi_f[i][l]) + kb * R(T.stoi_b[i][l])
    mw = [R(T.mw[l]) * R(1e3) for l in range(ns)]
    return (np.array([(made[l] - lost[l]) * mw[l] for l in range(ns)]),
            np.array([(made[l] + lost[l]) * mw[l] for l in range(ns)]))


def test_source_is_as_close_to_extended_precision_as_the_textbook_form():
    T = MX.load_mechanism(*MX.H2_AIR_FILES)
    ns, n_states = T.n_spec, 200
    case = pkg.cases.reacting_single_block(5, 5, 5, T, scheme=51, viscous_order=0)
    print(f"[gpu] fr chemical source of {n_states} uniform states", flush=True)
    s = MX.FrSolver(case, T)
    s.setup_mixing_layer()
    shape = s.shape(0, MX.FIELD_BV)[1:]
    met = np.zeros((9, *shape))
    met[0] = met[4] = met[8] = 1.0
    s.set_geometry(0, np.ones((1, *shape)), met)
    rng = np.random.default_rng(11)
    t = np.exp(rng.uniform(np.log(800.0), np.log(2800.0), n_states))
    Y = rng.dirichlet(np.ones(ns), n_states).T * 10.0 ** rng.uniform(-4, 0, (ns, n_states))
    Y[:, :] /= Y.sum(axis=0)
    mw = np.array(T.mw[:ns])
    rho = PATM / (RU * t * (Y / mw[:, None]).sum(axis=0))
    got = np.empty((ns, n_states))
    for q in range(n_states):
        bv = np.zeros((6, *shape))
        bv[0], bv[4], bv[5] = rho[q], PATM, t[q]
        s.set(0, MX.FIELD_BV, bv)
        s.set(0, MX.FIELD_SV, np.broadcast_to(Y[:, q, None, None, None], (ns, *shape)))
        s.initialize()
        s.compute_rhs(0)
        dq = s.get(0, MX.FIELD_DQ)[5:]
        assert np.all(dq == dq[:, :1, :1, :1]), q
        got[:, q] = dq[:, 2, 2, 2]
    s.close()
    exact, gross = _rates(T, rho, t, Y, np.longdouble)
    plain, _ = _rates(T, rho, t, Y, np.float64)
    some = gross[:, 0] > 0  # the bath gas takes no part
    err = [np.sqrt(np.mean((np.abs(x - exact)[some] / gross[some]).astype(float) ** 2, axis=1)) for x in (got, plain)]
    print("  gpu   ", " ".join(f"{e:.2e}" for e in err[0]), flush=True)
    print("  numpy ", " ".join(f"{e:.2e}" for e in err[1]), flush=True)
    assert np.all(got[~some] == 0)
    assert np.all(err[0] <= err[1]), err
