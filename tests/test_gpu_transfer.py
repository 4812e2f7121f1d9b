"""Copies of large host arrays through the pinned ring (csrc/transfer.cpp).

A MatMul of small whole numbers is exact in fp32, so an array that came up or
went down in the wrong place shows in the result.  Operand and result have the
same number of bytes: just below the line where the ring takes over, on it, one
row above, a ring's worth and a remainder, and one with partly filled chunks.
"""
import ctypes
import threading
import time

import numpy as np
import pytest

from gpu_util import note, require_hip

pytestmark = pytest.mark.gpu

MIB = 1 << 20


@pytest.fixture(scope="module")
def lc():
    return require_hip()


def product(lc, rows, seed, out=None):
    rng = np.random.default_rng(seed)
    a = rng.integers(-8, 9, (rows, 4)).astype(np.float32)
    b = rng.integers(-8, 9, (4, 4)).astype(np.float32)
    out = np.empty((rows, 4), np.float32) if out is None else out
    out[:] = np.nan
    s = lc.MatMulResidentSession(rows, 4, 4, "f32")
    s.start_into(a, b, out)
    s.finish_into(out=out)
    s.close()
    # not a @ b: two threads' matrix products at once have come out wrong in numpy's BLAS
    return out, sum(a[:, i : i + 1] * b[i : i + 1] for i in range(4))


@pytest.mark.parametrize("rows", [2 * MIB - 1, 2 * MIB, 2 * MIB + 1, 3 * MIB + 12345, 4 * MIB + 65537])
def test_large_arrays_arrive_whole(lc, rows):
    for seed in range(2):  # new inputs in the same ring
        got, want = product(lc, rows, seed)
        assert np.array_equal(got, want)


def test_two_threads_copy_at_once(lc):
    results = {}

    def work(i):
        results[i] = product(lc, 2 * MIB + 777 * i, 10 + i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(results) == 2
    for got, want in results.values():
        assert np.array_equal(got, want)


def test_upload_behind_queued_work(lc):
    """An upload that the stream reaches later arrives whole, and only the caller
    waits for the queue: a waiting thread spins, so the processor time stays
    below two cores (the caller's, and half again for the threads that copy once
    the queue has drained; all four spinning would take four)."""
    rng = np.random.default_rng(5)
    n = 4096
    busy = lc.MatMulResidentSession(n, n, n, "bf16")
    a = rng.standard_normal((n, n), dtype=np.float32)
    busy.start_into(a, a)
    busy.sync_into()
    rows = 2 * MIB + 5  # 32 MB and a remainder
    x = rng.integers(-8, 9, (rows, 4)).astype(np.float32)
    w = rng.integers(-8, 9, (4, 4)).astype(np.float32)
    s = lc.MatMulResidentSession(rows, 4, 4, "f32")
    s.start_into(x, w)
    out = np.empty((rows, 4), np.float32)
    s.finish_into(out=out)
    for _ in range(2):
        x = rng.integers(-8, 9, (rows, 4)).astype(np.float32)
        for _ in range(250):  # below the count at which a launch waits for the queue
            busy.run_into()
        wall, cpu = time.perf_counter(), time.process_time()
        s.start_into(x, w)
        wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
        note(f"[transfer] upload behind queued work: {wall * 1e3:.1f} ms, {cpu / wall:.2f} cores")
        assert wall > 0.01  # the queue was there
        assert cpu < 2 * wall
        s.finish_into(out=out)
        assert np.array_equal(out, sum(x[:, i : i + 1] * w[i : i + 1] for i in range(4)))
    s.close()
    busy.close()


def test_upload_to_new_buffers_keeps_its_rate(lc):
    """A new session's first kernels make its stream busy for a moment before its
    operands go up: they take as long as into the session's buffers later (the
    allocations and fills between them are 3% of it; half the rate would be twice)."""
    n = 8192
    a = np.ones((n, n), np.float32)
    fresh, again = [], []
    for _ in range(6):
        s = lc.MatMulResidentSession(n, n, n, "bf16")
        for times in (fresh, again):
            begin = time.perf_counter()
            s.start_into(a, a)
            times.append(time.perf_counter() - begin)
            s.sync_into()
        s.close()
    fresh, again = (sorted(times[1:])[2] for times in (fresh, again))  # the first call also times variants
    note(f"[transfer] 2 x 256 MB into new buffers {fresh * 1e3:.1f} ms, again {again * 1e3:.1f} ms")
    assert fresh < 1.6 * again


def test_pinned_result_buffer(lc):
    hip = ctypes.CDLL("libamdhip64.so.7")  # the runtime the backend has loaded
    rows = 2 * MIB + 5
    ptr = ctypes.c_void_p()
    assert hip.hipHostMalloc(ctypes.byref(ptr), ctypes.c_size_t(rows * 16), 0) == 0
    out = np.ctypeslib.as_array(ctypes.cast(ptr, ctypes.POINTER(ctypes.c_float)), (rows, 4))
    got, want = product(lc, rows, 3, out)
    same = np.array_equal(got, want)
    del got, out
    assert hip.hipHostFree(ptr) == 0
    assert same
