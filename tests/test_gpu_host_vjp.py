"""The host forms of the vector-Jacobian products, whose results of 4 MiB and more pass through the pinned staging
(copy_to_host in galx_api.hip), are bitwise their device forms, in the first call of a context and in later ones."""
import os

import numpy as np
import pytest

from galaexi_amd import mesh as M
from galaexi_amd import testcases as T

pytestmark = pytest.mark.gpu


# bytes of a result: 0.04 MB, 4.2 MB (just above the line), 22 MB
@pytest.mark.parametrize("N,nel", [(3, (3, 2, 2)), (4, (10, 10, 9)), (7, (11, 10, 10))])
def test_host_forms_equal_device_forms(N, nel):
    import torch

    from galaexi_amd import dg

    if len(os.sched_getaffinity(0)) <= 4:
        pytest.skip("hosts of few cores take the plain copy")
    print(f"case: N={N} {nel}", flush=True)
    lo, hi = (-1.0,) * 3, (1.0,) * 3
    m = M.box_mesh(nel, N, lo=lo, hi=hi, deform_amp=0.03, deform_phase=(0.1, 0.2, 0.3), NGeo=2)
    U, lam = (T.smooth_random(m.Elem_xGP, lo, hi, seed=s) for s in (1, 2))
    op = dg.DGOperator(N, form="split", riemann="lf", mu0=1e-3, R=1.0)
    op.set_mesh(m)
    op.set_state(U)

    def device(call, src=lam):
        t = torch.from_numpy(src.ravel(order="F").copy()).cuda()
        out = call(t)
        torch.cuda.synchronize()
        return (t if out is None else out).cpu().numpy().reshape(U.shape, order="F")

    def rhs_vjp(t):
        out = torch.empty_like(t)
        torch.cuda.synchronize()
        op.rhs_vjp_device(t.data_ptr(), out.data_ptr())
        return out

    def on(call):
        def run(t):
            torch.cuda.synchronize()
            call(t.data_ptr())

        return run

    for _ in range(2):
        assert np.array_equal(op.rhs_vjp(lam), device(rhs_vjp))
    got = op.step_vjp(0.0, 1e-4, lam)
    assert np.isfinite(got).all() and np.array_equal(got, device(on(lambda p: op.step_vjp_device(0.0, 1e-4, p))))
    op.forward_ckpt(0.0, 1e-4, 3, 2)
    for _ in range(2):
        assert np.array_equal(op.lserk_adjoint(lam), device(on(op.lserk_adjoint_device)))
    op.close()
