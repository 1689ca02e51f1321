"""A recorded run fills the stage inputs of its last segment for the reverse sweep: the gradient is bitwise the same whether
they come from the recorded run or from the sweep's recompute, for every checkpoint interval, for a second sweep over the
same recording, and after recordings of another length and VJPs of the current state in between."""
import numpy as np
import pytest

from galaexi_amd import mesh as M
from galaexi_amd import testcases as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,precision,source,nel", [(2, "fp64", False, (3, 2, 2)), (3, "fp64", True, (3, 2, 2)),
                                                    (3, "mixed", True, (3, 2, 2)), (5, "fp64", False, (3, 2, 2)),
                                                    (5, "mixed", False, (3, 2, 2)), (7, "fp64", False, (6, 5, 5))])
def test_gradient_does_not_depend_on_where_the_stages_come_from(N, precision, source, nel):
    from galaexi_amd import dg

    print(f"case: N={N} {precision} source={source} {nel}", flush=True)
    lo, hi = (-1.0, -1.0, -1.0), (1.0, 1.0, 1.0)
    m = M.box_mesh(nel, N, lo=lo, hi=hi, deform_amp=0.03, deform_phase=(0.1, 0.2, 0.3), NGeo=min(N, 3))
    U, lam, other = (T.smooth_random(m.Elem_xGP, lo, hi, seed=s) for s in (1, 2, 3))
    op = dg.DGOperator(N, form="split", riemann="lf", precision=precision, mu0=1e-3, R=1.0)
    op.set_mesh(m)
    if source:
        op.set_source(4, (0.3, 0.3, 0.3), m.Elem_xGP)
    final, grad = None, None
    for storage, every in (("steps", 2), ("stages", 1), ("stages", 2), ("stages", 5), ("stages", 3)):
        op.set_adjoint_storage(storage)
        op.set_state(other)
        op.forward_ckpt(0.0, 1e-4, 2, 1)  # another recording, whose stages the buffers hold
        op.set_state(U)
        op.forward_ckpt(0.1, 1e-4, 5, every)
        end = op.get_state()
        for sweep in range(2):
            got = op.lserk_adjoint(lam)
            assert np.isfinite(got).all() and np.array_equal(op.get_state(), end), (storage, every, sweep)
            grad = got if grad is None else grad
            assert np.array_equal(got, grad), (storage, every, sweep)
            op.rhs_vjp(lam)  # of the final state: leaves the recording alone
        final = end if final is None else final
        assert np.array_equal(end, final), (storage, every)
    op.set_state(U)
    op.TimeStepByLSERKW2(0.1, 1e-4, 5)
    assert np.array_equal(op.get_state(), final)
    op.close()
