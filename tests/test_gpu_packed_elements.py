"""GPU parity of the stage kernels of N = 1 and 2 on both sides of the line from which a workgroup takes several elements
(Pack in galx_kernels.hpp: 2048 elements; four of N = 1, two of N = 2), with full and partly filled last workgroups, on
curved meshes with rotated elements: Ut and one LSERK step against the FP64 oracle.

Bar: the FP64 bar of the parity tests, 1e-12 relative L2, plus four times what a change of U by one unit in the last
place does to the oracle's own result (the rounding that many elements along one direction amplify)."""
import numpy as np
import pytest

import oracle as O
from galaexi_amd import mesh as M
from galaexi_amd import testcases as T

pytestmark = pytest.mark.gpu

RIE = {"lf": O.RIEMANN_LF, "roeentropyfix": O.RIEMANN_ROEEF}
# below the line; on it; one and three elements left for the last workgroup of four, one for that of two
SIZES = [(6, 11, 31), (16, 16, 8), (11, 11, 17), (9, 11, 21)]


@pytest.mark.parametrize("form,riemann", [("split", "lf"), ("weak", "roeentropyfix")])
@pytest.mark.parametrize("nel", SIZES)
@pytest.mark.parametrize("N", [1, 2])
def test_packed_stage_kernels_vs_oracle(N, nel, form, riemann):
    from galaexi_amd import dg

    print(f"case: N={N} {nel} {form} {riemann}", flush=True)
    lo, hi = (-1.0, -1.0, -1.0), (1.0, 1.0, 1.0)
    m = M.box_mesh(nel, N, lo=lo, hi=hi, deform_amp=0.03, deform_phase=(0.13, 0.37, 0.71), NGeo=2,
                   rotations="random", seed=N)
    U = T.smooth_random(m.Elem_xGP, lo, hi, seed=N, kmax=1)
    gas = dict(mu0=2e-2, R=1.0, Pr=0.72, kappa=1.4)
    op = dg.DGOperator(N, form=form, riemann=riemann, **gas)
    op.set_mesh(m)
    op.set_state(U)
    ref = O.Operator(m, split=form == "split", riemann=RIE[riemann], **gas)
    ulp = np.random.default_rng(0).choice([-1.0, 1.0], U.shape) * np.finfo(float).eps
    U1 = np.asfortranarray(U * (1.0 + ulp))

    def check(got, want, want1, scale, what):
        err, own = (np.linalg.norm((a - want).ravel()) for a in (got, want1))
        assert err <= 1e-12 * np.linalg.norm(scale.ravel()) + 4.0 * own, (what, err, own, np.linalg.norm(scale.ravel()))

    Ut, Ur, Ur1 = op.DGTimeDerivative_weakForm(0.0), ref.rhs(U), ref.rhs(U1)
    for v in range(5):
        check(Ut[v], Ur[v], Ur1[v], Ur[v], v)
    dt, errType = op.CalcTimeStep()
    assert errType == 0
    op.TimeStepByLSERKW2(0.0, dt)
    Ug = op.get_state()
    op.close()
    W = []
    for start in (U, U1):
        W.append(np.asfortranarray(start.copy()))
        ref.lserk_step(W[-1], np.zeros_like(U, order="F"), 0.0, dt)
    check(Ug, W[0], W[1], W[0] - U, "step")
