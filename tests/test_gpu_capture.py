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
