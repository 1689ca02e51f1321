"""The manufactured source that the FP64 kernels add to the LSERK register (StageSource in galx_kernels.hpp: sin and cos
of omega*xs from a table, the angle sum with the stage time) against the source of a plain RHS evaluation (sincos of the
phase): U after a stage against U + b dt K with K = a K + Ut and Ut from DGTimeDerivative_weakForm, in every kernel that
updates the register.

Bar: the phase's rounding, (|omega xs| + |a t|) * 2 eps <= 4.5e-15 on [-1,1]^3 at t < 1, times the source's slope, at most
about 4 |S|, doubled for the two evaluations: 4e-14 of the source's part; and 8 eps of every term of the sum."""
import numpy as np
import pytest

from galaexi_amd import mesh as M
from galaexi_amd import testcases as T

pytestmark = pytest.mark.gpu

ADV = (0.3, 0.3, 0.3)
EPS = np.finfo(float).eps
RKA = [0.0, 567301805773.0 / 1357537059087.0, 2404267990393.0 / 2016746695238.0]
RKB = [1432997174477.0 / 9575080441755.0, 5161836677717.0 / 13612068292357.0, 1720146321549.0 / 2090206949498.0]
RKC = [0.0, RKB[0], 2526269341429.0 / 6820363962896.0]


# packed, one element per workgroup, planes
@pytest.mark.parametrize("N,nel,form,riemann", [
    (1, (13, 13, 13), "split", "lf"), (2, (13, 13, 13), "weak", "roeentropyfix"), (2, (3, 2, 2), "split", "roe"),
    (3, (4, 3, 2), "split", "roeentropyfix"), (4, (7, 6, 5), "weak", "lf"), (5, (4, 3, 2), "split", "roe"),
    (5, (9, 5, 4), "split", "roeentropyfix"), (7, (6, 5, 5), "split", "lf"), (8, (6, 5, 4), "split", "lf"),
    (9, (2, 2, 2), "weak", "roe"), (11, (2, 2, 2), "split", "roeentropyfix")])
def test_source_of_a_stage_equals_that_of_a_plain_rhs(N, nel, form, riemann):
    from galaexi_amd import dg

    print(f"case: N={N} {nel} {form} {riemann}", flush=True)
    m = M.box_mesh(nel, N, lo=(-1.0,) * 3, hi=(1.0,) * 3)
    op = dg.DGOperator(N, form=form, riemann=riemann, mu0=1e-3, R=287.058, Pr=0.72, kappa=1.4)
    op.set_mesh(m)
    rng = np.random.default_rng(N)
    t = 0.37
    norm = lambda x: np.linalg.norm(np.ravel(x))
    for case in T.SOURCE_FUNCS:
        U = T.synthetic_wave(case, m.Elem_xGP, t, ADV)
        U = np.asfortranarray(U * (1.0 + 1e-3 * rng.standard_normal(U.shape)))
        op.set_source(case, ADV, m.Elem_xGP)
        op.set_state(U)
        dt, errType = op.CalcTimeStep()
        assert errType == 0
        # a single large stage, whose increment is of the size of U, then three of a step
        for h, stages in ((1.0, 1), (dt, 3)):
            op.set_state(U)
            cur, K = U, np.zeros_like(U)
            for s in range(stages):
                ts = t + RKC[s] * h
                op.set_source(0, ADV)
                Ut0 = op.DGTimeDerivative_weakForm(ts)
                op.set_source(case, ADV, m.Elem_xGP)
                Ut = op.DGTimeDerivative_weakForm(ts)
                old, K = K, -RKA[s] * K + Ut
                op.lserk_stage(t, h, s + 1)
                got, want = op.get_state(), cur + RKB[s] * h * K
                size = norm(cur) + norm(got) + RKB[s] * h * (norm(old) + norm(Ut) + norm(Ut0))
                bar = 4e-14 * RKB[s] * h * norm(Ut - Ut0) + 8 * EPS * size
                assert norm(got - want) <= bar, (case, h, s, norm(got - want), bar)
                cur = got
    op.close()
