"""A context that has run before behaves like a new one after galx_set_state: its LSERK register counts as zero whatever its
memory holds (a stage with a non-zero register coefficient as the first one included), the mixed form's offsets are those
of the new state, and the time step's error flag does not outlast the call that raised it.  Bitwise."""
import numpy as np
import pytest

from galaexi_amd import mesh as M
from galaexi_amd import testcases as T

pytestmark = pytest.mark.gpu

ADV = (0.3, 0.3, 0.3)


def context(m, precision, source):
    from galaexi_amd import dg

    op = dg.DGOperator(m.N, form="split", riemann="lf", precision=precision, mu0=1e-3, R=1.0)
    op.set_mesh(m)
    if source:
        op.set_source(4, ADV, m.Elem_xGP)
    return op


@pytest.mark.parametrize("N,precision,source,nel", [(2, "fp64", False, (3, 2, 2)), (3, "fp64", True, (3, 2, 2)),
                                                    (3, "mixed", True, (3, 2, 2)), (5, "mixed", False, (3, 2, 2)),
                                                    (7, "fp64", False, (2, 2, 2)), (7, "fp64", False, (7, 5, 4)),
                                                    (11, "fp64", True, (2, 2, 2))])
def test_used_context_equals_new_one(N, precision, source, nel):
    print(f"case: N={N} {precision} source={source} {nel}", flush=True)
    lo, hi = (-1.0, -1.0, -1.0), (1.0, 1.0, 1.0)
    m = M.box_mesh(nel, N, lo=lo, hi=hi, deform_amp=0.03, deform_phase=(0.1, 0.2, 0.3), NGeo=min(N, 3))
    U, V = (T.smooth_random(m.Elem_xGP, lo, hi, seed=s) for s in (1, 2))
    used, new = context(m, precision, source), context(m, precision, source)
    bad = U.copy(order="F")
    bad[0] = -bad[0]
    used.set_state(bad)
    assert used.CalcTimeStep()[1] == 1
    used.TimeStepByLSERKW2(0.0, 1e-4, 2)  # leaves NaN in the state and the register
    used.set_state(V)
    used.TimeStepByLSERKW2(0.0, 1e-4, 2)
    for op in (used, new):
        op.set_state(U)
    assert used.CalcTimeStep() == new.CalcTimeStep() and new.CalcTimeStep()[1] == 0
    for stage in (3, 4, 1, 2):  # the first one has a non-zero register coefficient
        for op in (used, new):
            op.lserk_stage(0.1, 1e-4, stage)
        a, b = used.get_state(), new.get_state()
        assert np.isfinite(b).all() and np.array_equal(a, b), stage
    used.close()
    new.close()
