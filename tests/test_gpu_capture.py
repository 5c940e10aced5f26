"""Calls that wait for a result on a stream that is being captured: refused
at once, with the capture ended (the runtime keeps that stream for good);
other contexts go on.
"""
import ctypes
import time

import numpy as np
import pytest

from gip_amd import cavity, hip

pytestmark = pytest.mark.gpu

THREAD_LOCAL = 1


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


@pytest.mark.parametrize("call", ["dot", "cfl", "solve", "solve_noalloc"])
def test_a_result_under_capture_is_refused_at_once(dev, call):
    hiprt = ctypes.CDLL("libamdhip64.so")
    other, dev = dev, hip.Device(0)
    c = cavity.generate(16, gamma=1e-2, ops=cavity.OP_BITS["L"])
    A = hip.Matrix.from_csr(dev, c.op("L"))
    solver = hip.PCG(A, c.n_all)
    v = np.zeros(c.n_all)
    v[:c.n_inner] = cavity.rhs_normal(c.n_inner, 1)
    b, x, z = dev.to_device(v), dev.array(c.n_all), dev.to_device(np.zeros(c.n_all))
    one = dev.to_device(np.ones(c.n_all))
    calls = {"dot": lambda: hip.dot(b, b), "cfl": lambda: hip.cfl(b, b, b, one, c.n_inner, 1e-2, 1.0),
             "solve": lambda: solver.solve(b, x, z, maxit=8).iters,
             "solve_noalloc": lambda: hip.pcg_solve_noalloc(A, c.n_all, b, x, z, maxit=8).iters}
    want = calls[call]()
    stream, graph = ctypes.c_void_p(hip.lib().gip_stream(dev.ctx)), ctypes.c_void_p()
    assert hiprt.hipStreamBeginCapture(stream, THREAD_LOCAL) == 0
    t0 = time.perf_counter()
    with pytest.raises(hip.HipError):
        calls[call]()
    took = time.perf_counter() - t0
    assert hiprt.hipStreamEndCapture(stream, ctypes.byref(graph)) != 0 and not graph.value
    dev.close()
    hiprt.hipGetLastError()
    print(f"[capture {call}] refused after {1e3 * took:.2f} ms (uncaptured result {want})", flush=True)
    # a wait that spins asks for the stream after about 40 ms
    assert took < 0.02
    ones = other.to_device(np.ones(1000))
    assert hip.dot(ones, ones) == 1000.0


def symmetric_without_repeats(shape, seed=1):
    """A cavity Laplacian scaled to (s_i s_j) a_ij: bitwise symmetric, no two rows alike."""
    c = cavity.generate(*shape, gamma=1e-2, ops=cavity.OP_BITS["L"])
    L = c.op("L")
    row = np.repeat(np.arange(L.nrows), np.diff(L.rowptr))
    s = 1.0 + 0.1 * np.random.default_rng(seed).random(max(L.nrows, int(L.col.max()) + 1))
    return L.rowptr.copy(), L.col.copy(), (s[row] * s[L.col]) * L.val, L.nrows


def test_solves_follow_values_that_a_graph_changes(dev):
    """A replayed graph changes an operator's values without the host's doing: the symmetric form made before it
    is not used any more."""
    torch = pytest.importorskip("torch")
    rowptr, col, val, n = symmetric_without_repeats((96, 96, 64))
    nall, nnz = max(n, int(col.max()) + 1), val.size
    A = hip.Matrix(dev, rowptr, col, val, nrows=n)
    b, x, z = dev.to_device(cavity.rhs_normal(n, 3)), dev.array(nall), dev.to_device(np.zeros(nall))
    solver = hip.PCG(A, nall)
    solver.solve(b, x, z, maxit=3)
    assert A.sym_state()[0] == 1
    ident = hip.Matrix(dev, np.arange(nnz + 1), np.arange(nnz), np.ones(nnz), ncols=nnz, fmt=hip.FMT_CSR)
    other = val.copy()
    other[col != np.repeat(np.arange(n), np.diff(rowptr))] *= 0.5
    dv = dev.to_device(other)
    stream = torch.cuda.ExternalStream(hip.lib().gip_stream(dev.ctx))
    change = torch.cuda.CUDAGraph()
    with torch.cuda.graph(change, stream=stream, capture_error_mode="thread_local"):
        ident.spmv_vals(dv, A)
    for _ in range(2):
        # made again from values set by the host, then changed by a replay
        A.set_values(val)
        solver.solve(b, x, z, maxit=3)
        with torch.cuda.stream(stream):
            change.replay()
        solver.solve(b, x, z, maxit=12)
        got = x.download()
        F = hip.Matrix(dev, rowptr, col, other, nrows=n, sym=False)
        full = hip.PCG(F, nall)
        full.solve(b, x, z, maxit=12)
        assert np.array_equal(got, x.download())
