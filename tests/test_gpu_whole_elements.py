"""The stage kernels of one element per workgroup (k_lift, k_rhs) on meshes above the line up to which FP64 meshes take the
plane kernels (1024 planes, use_planes in galx_kernels_plane.hpp): every degree, form and solver, on curved meshes with
rotated elements, Ut, dt and two LSERK steps against the FP64 oracle; free-stream preservation; and the mixed form at N = 3
around the lines from which k_rhs (1536 elements) and k_lift (4096) take an element with 64 threads (FaceBlock).

Bars.  FP64: that of the parity tests, 1e-12 relative L2, plus four times what a change of U by one unit in the last place
does to the oracle's own result.  Free stream: that of the parity tests.  Mixed: that of the parity tests, 1e-4 relative L2
of Ut, and as much of the change of U over a step, a sum of such Ut."""
import numpy as np
import pytest

import oracle as O
from galaexi_amd import mesh as M
from galaexi_amd import testcases as T

pytestmark = pytest.mark.gpu

RIE = {"lf": O.RIEMANN_LF, "roe": O.RIEMANN_ROE, "roeentropyfix": O.RIEMANN_ROEEF}
LO, HI = (-1.0, -1.0, -1.0), (1.0, 1.0, 1.0)
GAS = dict(mu0=2e-2, R=1.0, Pr=0.72, kappa=1.4)
ABOVE = {4: (7, 6, 5), 5: (7, 5, 5), 6: (6, 5, 5), 7: (5, 9, 3), 8: (6, 5, 4), 9: (7, 5, 3)}
# with 64-thread workgroups in neither kernel, in k_rhs only (just above its line, and on that of k_lift), in both
MIXED = [(16, 12, 8), (12, 12, 11), (16, 16, 16), (17, 16, 16)]


def curved(nel, N):
    return M.box_mesh(nel, N, lo=LO, hi=HI, deform_amp=0.03, deform_phase=(0.13, 0.37, 0.71), NGeo=2, rotations="random",
                      seed=N)


def context(m, form, riemann, U, **kw):
    from galaexi_amd import dg

    op = dg.DGOperator(m.N, form=form, riemann=riemann, CFLScale=0.9, DFLScale=0.9, **dict(GAS, **kw))
    op.set_mesh(m)
    op.set_state(U)
    return op


def two_steps(ref, U, dt):
    W, K = np.asfortranarray(U.copy()), np.zeros_like(U, order="F")
    for s in range(2):
        ref.lserk_step(W, K, s * dt, dt)
    return W


def test_sizes_lie_above_the_line():
    assert all(int(np.prod(nel)) * (N + 1) > 1024 for N, nel in ABOVE.items())


@pytest.mark.parametrize("riemann", sorted(RIE))
@pytest.mark.parametrize("form", ["split", "weak"])
@pytest.mark.parametrize("N", sorted(ABOVE))
def test_fp64_vs_oracle(N, form, riemann):
    print(f"case: N={N} {ABOVE[N]} {form} {riemann}", flush=True)
    m = curved(ABOVE[N], N)
    U = T.smooth_random(m.Elem_xGP, LO, HI, seed=N, kmax=1)
    op = context(m, form, riemann, U)
    ref = O.Operator(m, split=form == "split", riemann=RIE[riemann], **GAS)
    ulp = np.random.default_rng(0).choice([-1.0, 1.0], U.shape) * np.finfo(float).eps
    U1 = np.asfortranarray(U * (1.0 + ulp))

    def check(got, want, want1, scale, what):
        err, own = (np.linalg.norm((a - want).ravel()) for a in (got, want1))
        assert err <= 1e-12 * np.linalg.norm(scale.ravel()) + 4.0 * own, (what, err, own, np.linalg.norm(scale.ravel()))

    Ut, Ur, Ur1 = op.DGTimeDerivative_weakForm(0.0), ref.rhs(U), ref.rhs(U1)
    for v in range(5):
        check(Ut[v], Ur[v], Ur1[v], Ur[v], v)
    dt, errType = op.CalcTimeStep()
    dt_ref, err_ref, _, _ = ref.calc_dt(U, 0.9, 0.9)
    assert errType == 0 and err_ref == 0 and abs(dt - dt_ref) <= 1e-14 * dt_ref
    op.TimeStepByLSERKW2(0.0, dt, nSteps=2)
    Ug = op.get_state()
    op.close()
    W, W1 = two_steps(ref, U, dt), two_steps(ref, U1, dt)
    check(Ug, W, W1, W - U, "steps")


@pytest.mark.parametrize("form", ["split", "weak"])
@pytest.mark.parametrize("N", sorted(ABOVE))
def test_freestream(N, form):
    print(f"case: free stream N={N} {ABOVE[N]} {form}", flush=True)
    m = curved(ABOVE[N], N)
    U = T.freestream(m.Elem_xGP)
    op = context(m, form, "roeentropyfix", U, mu0=1e-3)
    Ut = op.DGTimeDerivative_weakForm()
    op.close()
    ref = O.Operator(m, split=form == "split", riemann=O.RIEMANN_ROEEF, **dict(GAS, mu0=1e-3)).rhs(U)
    # round-off scale of the operator: sJ * |U| * (N+1)^2 (line sums of D entries of size ~N^2)
    scale = np.abs(m.sJ).max() * np.abs(U).max() * (N + 1) ** 2
    assert np.abs(Ut).max() <= 1e-13 * scale
    assert np.abs(Ut).max() <= 30 * max(np.abs(ref).max(), 1e-15 * scale)


@pytest.mark.parametrize("form,riemann", [("split", "lf"), ("weak", "roe"), ("split", "roeentropyfix")])
@pytest.mark.parametrize("nel", MIXED)
def test_mixed_n3_vs_oracle(nel, form, riemann):
    print(f"case: mixed N=3 {nel} {form} {riemann}", flush=True)
    m = curved(nel, 3)
    U = T.smooth_random(m.Elem_xGP, LO, HI, seed=3)
    op = context(m, form, riemann, U, precision="mixed")
    ref = O.Operator(m, split=form == "split", riemann=RIE[riemann], **GAS)
    Ut, Ur = op.DGTimeDerivative_weakForm(0.0), ref.rhs(U)
    for v in range(5):
        assert np.linalg.norm((Ut[v] - Ur[v]).ravel()) <= 1e-4 * np.linalg.norm(Ur[v].ravel()), v
    dt, errType = op.CalcTimeStep()
    assert errType == 0
    op.TimeStepByLSERKW2(0.0, dt, nSteps=2)
    Ug = op.get_state()
    op.close()
    W = two_steps(ref, U, dt)
    assert np.linalg.norm((Ug - W).ravel()) <= 1e-4 * np.linalg.norm((W - U).ravel())
