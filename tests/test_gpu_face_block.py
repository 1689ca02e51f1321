"""The stage kernels whose workgroups take all face nodes in one pass (FaceBlock in galx_kernels.hpp: k_lift at N = 3 and 4,
k_rhs there up to 1536 and 3072 elements) against the oracle, on both sides of the lines of k_rhs, FP64, on curved meshes
with rotated elements.

Bar (FP64): that of the parity tests, 1e-12 relative L2, plus four times what a change of U by one unit in the last place
does to the oracle's own result."""
import numpy as np
import pytest

import oracle as O
from galaexi_amd import mesh as M
from galaexi_amd import testcases as T

pytestmark = pytest.mark.gpu

RIE = {"lf": O.RIEMANN_LF, "roe": O.RIEMANN_ROE, "roeentropyfix": O.RIEMANN_ROEEF}
# below the line, on it, above it; N = 4 above the plane kernels' range
SIZES = {3: [(3, 2, 2), (16, 12, 8), (29, 53, 1)], 4: [(7, 6, 5), (16, 16, 12), (7, 439, 1)]}


@pytest.mark.parametrize("form,riemann", [("split", "roeentropyfix"), ("weak", "roe")])
@pytest.mark.parametrize("N,nel", [(N, nel) for N in SIZES for nel in SIZES[N]])
def test_face_block_vs_oracle(N, nel, form, riemann):
    from galaexi_amd import dg

    print(f"case: N={N} {nel} {form} {riemann}", flush=True)
    lo, hi = (-1.0, -1.0, -1.0), (1.0, 1.0, 1.0)
    m = M.box_mesh(nel, N, lo=lo, hi=hi, deform_amp=0.03, deform_phase=(0.13, 0.37, 0.71), NGeo=2,
                   rotations="random" if min(nel) > 1 else None, seed=N)
    U = T.smooth_random(m.Elem_xGP, lo, hi, seed=N, kmax=1)
    gas = dict(mu0=2e-2, R=1.0, Pr=0.72, kappa=1.4)
    op = dg.DGOperator(N, form=form, riemann=riemann, **gas)
    op.set_mesh(m)
    op.set_state(U)
    ref = O.Operator(m, split=form == "split", riemann=RIE[riemann], **gas)
    ulp = np.random.default_rng(0).choice([-1.0, 1.0], U.shape) * np.finfo(float).eps
    U1 = np.asfortranarray(U * (1.0 + ulp))
    Ut, Ur, Ur1 = op.DGTimeDerivative_weakForm(0.0), ref.rhs(U), ref.rhs(U1)
    for v in range(5):
        err, own = np.linalg.norm((Ut[v] - Ur[v]).ravel()), np.linalg.norm((Ur1[v] - Ur[v]).ravel())
        assert err <= 1e-12 * np.linalg.norm(Ur[v].ravel()) + 4.0 * own, (v, err, own)
    op.close()
