"""The library's host code with the HIP runtime replaced (tests/native/hip_stub.cpp): results on their way to pageable host
arrays.  Device memory holds the indices of its doubles, and so does the state handed in; no kernel runs, so a result is right
if it is arange.  A copy that nobody waits for never arrives.  Each scenario runs in a process of its own, with the stub ahead of the HIP runtime."""
import os
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PRELUDE = """
import ctypes, sys, time
import numpy as np
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.modules["torch"] = None  # its HIP runtime would be loaded ahead of the stub
from galaexi_amd import _lib, dg, mesh as M

def fail(name, nth):
    stub.stub_fail(name.encode(), ctypes.c_long(nth))

def calls(name):
    return stub.stub_calls(name.encode())

def context(N, nel, precision="fp64"):
    op = dg.DGOperator(N, form="split", riemann="lf", precision=precision, mu0=1e-3, R=1.0)
    m = M.box_mesh(nel, N, lo=(-1.0,) * 3, hi=(1.0,) * 3)
    op.set_mesh(m)
    op.set_state(np.arange(5.0 * (N + 1) ** 3 * m.nElems).reshape((5, N + 1, N + 1, N + 1, m.nElems), order="F"))
    return op

def right(U):
    return np.array_equal(U.ravel(order="F"), np.arange(U.size))

def refused(f, *a):
    try:
        f(*a)
    except _lib.GalxError as e:
        return str(e)
    raise AssertionError("not refused")

CHUNKS = 12  # of 2 MiB, over 4 slots: the results of BIG
BIG = (4, (11, 21, 21))
assert 11 * 21 * 21 * 125 * 40 > (CHUNKS - 1) << 21 and 11 * 21 * 21 * 125 * 40 < CHUNKS << 21
"""


@pytest.fixture(scope="session")
def stub(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("hip_stub") / "libhip_stub.so")
    src = os.path.join(ROOT, "tests", "native", "hip_stub.cpp")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-o", out, src], check=True)
    return out


def run(stub, body):
    env = dict(os.environ, OMP_NUM_THREADS="1", OPENBLAS_NUM_THREADS="1")
    res = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(body), stub], cwd=ROOT, env=env, text=True,
                         capture_output=True, timeout=100)
    assert res.returncode == 0, res.stdout + res.stderr


needs_cores = pytest.mark.skipif(len(os.sched_getaffinity(0)) <= 4, reason="hosts of few cores take the plain copy")


@needs_cores
def test_large_results_go_through_the_chunks(stub):
    run(stub, """
        op = context(*BIG)
        for _ in range(3):
            n = calls("hipMemcpyAsync")
            assert right(op.get_state())
            assert calls("hipMemcpyAsync") - n == CHUNKS
        op.close()
        op = context(4, (10, 9, 9))  # 4.05 MB, below 4 MiB: one plain copy
        n = calls("hipMemcpyAsync")
        assert right(op.get_state()) and calls("hipMemcpyAsync") - n == 1
    """)


@needs_cores
def test_waiting_for_queued_work_takes_no_processor_time(stub):
    """Copies start when the work queued before them is done; until then nothing may spin.  Half a core is the bar: the stub
    sleeps, and copying the 24 MB takes some 10 ms."""
    run(stub, """
        op = context(*BIG)
        op.get_state()
        for get in (op.get_state, lambda: op.get_gradients()[0]):
            stub.stub_busy(400000)
            cpu, wall = time.process_time(), time.perf_counter()
            U = get()
            cpu, wall = time.process_time() - cpu, time.perf_counter() - wall
            assert right(U) and wall > 0.4 and cpu < 0.2, (cpu, wall)
    """)


@needs_cores
@pytest.mark.parametrize("spare_mb", [12, 28])
def test_plain_copy_where_threads_cannot_be_created(stub, spare_mb):
    """Address space for the stacks of one or none of the four threads, and of two or three."""
    run(stub, f"""
        import resource
        op = context(*BIG)
        U = np.zeros(op._shape(), order="F")
        used = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
        old = resource.getrlimit(resource.RLIMIT_AS)
        n = calls("hipMemcpyAsync")
        resource.setrlimit(resource.RLIMIT_AS, (used + ({spare_mb} << 20), old[1]))
        rc = _lib.lib().galx_get_state(op._h, dg._dptr(U))
        resource.setrlimit(resource.RLIMIT_AS, old)
        assert rc == 0 and right(U) and stub.stub_pending() == 0
        assert calls("hipMemcpyAsync") - n in (1, 5)  # the plain copy alone, or after a first round of the slots
    """)


@needs_cores
@pytest.mark.parametrize("call,nth", [("hipMemcpyAsync", 3), ("hipMemcpyAsync", 9), ("hipEventRecord", 2),
                                      ("hipEventSynchronize", 1), ("hipEventSynchronize", 7)])
def test_no_copy_outlives_a_failed_call(stub, call, nth):
    """A copy still under way would write into the slots of the next call, or into an array the caller has freed."""
    run(stub, f"""
        op = context(*BIG)
        assert right(op.get_state())
        fail("{call}", {nth})
        assert "stub error" in refused(op.get_state)
        assert stub.stub_pending() == 0
        stub.hipGetLastError()  # the runtime keeps it until it is asked
        assert right(op.get_state()) and stub.stub_pending() == 0
    """)


def test_no_plain_copy_outlives_a_failed_call(stub):
    run(stub, """
        op = context(4, (3, 3, 3))
        fail("hipMemcpyAsync", 2)
        assert "stub error" in refused(op.get_gradients)
        assert stub.stub_pending() == 0
    """)


@pytest.mark.parametrize("N,precision,launch", [(3, "fp64", 1), (3, "mixed", 1), (3, "mixed", 2), (11, "fp64", 1)])
def test_failed_set_state_leaves_no_state(stub, N, precision, launch):
    """The state's planes and its traces, offsets and register belong together: after a call that wrote only some of them
    there is nothing to step from."""
    run(stub, f"""
        op = context({N}, (2, 2, 2), "{precision}")
        U = np.ones(op._shape(), order="F")
        op.TimeStepByLSERKW2(0.0, 1e-3)
        fail("hipLaunchKernel", {launch})
        assert "stub error" in refused(op.set_state, U)
        for call in (lambda: op.TimeStepByLSERKW2(0.0, 1e-3), lambda: op.lserk_stage(0.0, 1e-3, 1), op.get_state,
                     op.CalcTimeStep, op.get_gradients, op.rhs_only):
            assert any(why in refused(call) for why in ("set_state first", "no state"))
        op.set_state(U)
        op.TimeStepByLSERKW2(0.0, 1e-3)
    """)


def test_failed_recompute_is_not_taken_for_the_stages(stub):
    """The sweep counts the stage inputs of a segment as there once their kernels have been launched: the sweep after a failed
    one launches what one without the failure does."""
    run(stub, """
        op = context(3, (2, 2, 2))
        lam = np.ones(op._shape(), order="F")
        op.forward_ckpt(0.0, 1e-3, 4, 2)
        op.lserk_adjoint(lam)  # the last segment's stages come from the recorded run; it leaves those of the first one
        n = calls("hipLaunchKernel")
        op.lserk_adjoint(lam)
        full = calls("hipLaunchKernel") - n
        fail("hipLaunchKernel", 10)  # in the recompute of the last segment
        assert "stub error" in refused(op.lserk_adjoint, lam)
        n = calls("hipLaunchKernel")
        op.lserk_adjoint(lam)
        assert calls("hipLaunchKernel") - n == full
    """)


@needs_cores
def test_first_results_allocate_nothing_but_their_scratch(stub):
    """The pinned chunks are those that galx_set_mesh staged the geometry through: pinning them at the first result took
    longer than the chunks save there."""
    run(stub, """
        for N, nel in (BIG, (7, (9, 5, 4)), (11, (4, 3, 2))):
            op = context(N, nel)
            pinned, copies = calls("hipHostMalloc"), calls("hipMemcpyAsync")
            g = op.get_gradients(5)
            assert calls("hipHostMalloc") == pinned and calls("hipMemcpyAsync") - copies >= 3
            n = g[0].size
            assert all(np.array_equal(a.ravel(order="F"), np.arange(d * n, (d + 1) * n)) for d, a in enumerate(g))
            op.close()
        n = calls("hipHostMalloc")
        context(7, (3, 3, 3)).close()  # its largest result stays below 4 MiB: two buffers for the geometry, dt's two doubles
        assert calls("hipHostMalloc") - n == 3
    """)


def test_failed_set_mesh_leaves_nothing_pinned(stub):
    run(stub, """
        op = dg.DGOperator(7, form="split", riemann="lf", mu0=1e-3, R=1.0)
        m = M.box_mesh((9, 5, 4), 7, lo=(-1.0,) * 3, hi=(1.0,) * 3)
        for call, nth in (("hipHostMalloc", 1), ("hipMemcpyAsync", 1), ("hipMemcpyAsync", 7), ("hipEventRecord", 2)):
            held = calls("hipHostMalloc") - calls("hipHostFree")
            fail(call, nth)
            assert "stub error" in refused(op.set_mesh, m) or call == "hipHostMalloc"
            stub.hipGetLastError()
            assert stub.stub_pending() == 0
            assert calls("hipHostMalloc") - calls("hipHostFree") - (call == "hipHostMalloc") == held
        op.set_mesh(m)
    """)
