"""Results copied to host arrays through the pinned staging (copy_to_host in galx_api.hip, from 4 MiB on, in 2 MiB chunks
over 4 slots) are bitwise those of the plain copy, which pinned host arrays take: sizes below the line, of one chunk and a
remainder, and of more chunks than slots; from several threads with a context each."""
import threading

import numpy as np
import pytest

from galaexi_amd import mesh as M
from galaexi_amd import testcases as T

pytestmark = pytest.mark.gpu


def context(N, nel, seed=1):
    from galaexi_amd import dg

    lo, hi = (-1.0,) * 3, (1.0,) * 3
    m = M.box_mesh(nel, N, lo=lo, hi=hi)
    op = dg.DGOperator(N, form="split", riemann="lf", mu0=1e-3, R=1.0)
    op.set_mesh(m)
    op.set_state(T.smooth_random(m.Elem_xGP, lo, hi, seed=seed))
    return op


def pinned(shape):
    import torch

    t = torch.empty(int(np.prod(shape)), dtype=torch.float64).pin_memory()
    return t, t.numpy().reshape(shape, order="F")


# bytes of the state: 0.04 MB, 4.0 (below 4 MiB), 4.2 (above), 22 (more chunks than slots)
@pytest.mark.parametrize("N,nel", [(3, (3, 2, 2)), (4, (10, 9, 9)), (4, (10, 9, 9 + 1)), (7, (11, 10, 10))])
def test_staged_results_equal_plain_copies(N, nel):
    from galaexi_amd import dg
    from galaexi_amd._lib import lib

    print(f"case: N={N} {nel}", flush=True)
    op = context(N, nel)
    for _ in range(2):
        U, g = op.get_state(), op.get_gradients()
        tU, pU = pinned(U.shape)
        assert lib().galx_get_state(op._h, dg._dptr(pU)) == 0
        assert np.array_equal(U, pU)
        pg = [pinned(a.shape) for a in g]
        assert lib().galx_get_lifted_gradients(op._h, 4, *[dg._dptr(a) for _, a in pg]) == 0
        assert all(np.array_equal(a, b) for a, (_, b) in zip(g, pg))
        dt, _ = op.CalcTimeStep()
        op.TimeStepByLSERKW2(0.0, dt)
    op.close()


def test_several_threads():
    ops = [context(5, (10, 9, 8), seed=s) for s in range(3)]
    want = [op.get_state() for op in ops]
    got = [[None] * 4 for _ in ops]

    def run(i):
        for k in range(4):
            got[i][k] = ops[i].get_state()

    ts = [threading.Thread(target=run, args=(i,)) for i in range(len(ops))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert all(np.array_equal(g, w) for gs, w in zip(got, want) for g in gs)
    for op in ops:
        op.close()
