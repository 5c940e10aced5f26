"""gip_sync: it returns when the work queued before it is done, for one thread
and for several on a context, without leaving the stream unusable.
"""
import threading

import numpy as np
import pytest

from gip_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


class _Raw:
    def __init__(self, a):
        self.__cuda_array_interface__ = {"shape": (a.n,), "typestr": a.dtype.str, "data": (a.ptr.value, False),
                                         "version": 2}


def test_work_queued_before_is_done(dev):
    """100 updates of 64 MB (some milliseconds), read on another stream right after the call."""
    torch = pytest.importorskip("torch")
    n = 1 << 23
    x, y = dev.to_device(np.ones(n)), dev.to_device(np.zeros(n))
    view = torch.as_tensor(_Raw(y), device="cuda")
    other = torch.cuda.Stream()
    for rep in range(1, 6):
        for _ in range(100):
            hip.axpy(1.0, x, y)
        dev.sync()
        with torch.cuda.stream(other):
            low, high = view.min().item(), view.max().item()
        assert low == high == 100.0 * rep


def test_several_threads_wait_on_one_context(dev):
    n, calls, errors = 1 << 16, 400, []
    x, y = dev.to_device(np.ones(n)), [dev.to_device(np.zeros(n)) for _ in range(4)]

    def work(mine):
        try:
            for _ in range(calls):
                hip.axpy(1.0, x, mine)
                dev.sync()
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(v,)) for v in y]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not errors and not any(t.is_alive() for t in threads)
    dev.sync()
    for v in y:
        assert np.array_equal(v.download(), np.full(n, float(calls)))


def test_an_idle_stream_costs_no_kernel(dev):
    """After a copy to the host, which drains the stream, the call returns at once (0.4 us; a kernel and its wait
    6.1); after a host result it waits for a kernel of its own (6.4 more than the result, the runtime's wait 9.6)."""
    import time

    x = dev.to_device(np.ones(1000))

    def best(call, reps=300):
        times = []
        for _ in range(5):
            t0 = time.perf_counter()
            for _ in range(reps):
                call()
            times.append((time.perf_counter() - t0) / reps)
        return 1e6 * min(times)

    x.download()
    idle = best(dev.sync)
    one, both = best(lambda: hip.dot(x, x)), best(lambda: (hip.dot(x, x), dev.sync()))
    print(f"[gip_sync] idle {idle:.2f} us, dot {one:.2f}, dot and gip_sync {both:.2f}", flush=True)
    assert idle < 3.0 and both - one < 8.5
