"""The bf16 planes that fp32 sessions keep beside their operands (1.5 times a
GEMM's operands, 4.5 times an attention tensor) give way when memory runs out:
sessions that fit a device's memory without planes fit it together, and every
one of them still answers.
"""
import contextlib
import ctypes

import numpy as np
import pytest

from gpu_util import note, require_hip

pytestmark = pytest.mark.gpu

MIB = 1 << 20


@pytest.fixture(scope="module")
def lc():
    return require_hip()


@contextlib.contextmanager
def only(hip, left):
    """Device memory taken but for `left` bytes."""
    held = []
    try:
        while True:
            free, total = ctypes.c_size_t(), ctypes.c_size_t()
            assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
            size = min(free.value - left, 32 << 30) // (2 * MIB) * (2 * MIB)
            if size <= 0:
                break
            ptr = ctypes.c_void_p()
            assert hip.hipMalloc(ctypes.byref(ptr), ctypes.c_size_t(size)) == 0
            held.append(ptr)
        yield
    finally:
        for ptr in held:
            assert hip.hipFree(ptr) == 0


def test_planes_give_way_to_another_session(lc):
    hip = ctypes.CDLL("libamdhip64.so.7")  # the runtime the backend has loaded
    n = 8192
    rng = np.random.default_rng(21)
    a, b = (rng.standard_normal((n, n), dtype=np.float32) for _ in range(2))
    rows = [0, 4095, n - 1]
    want = a[rows].astype(np.float64) @ b.astype(np.float64)

    def check(got):
        assert np.linalg.norm(got.reshape(n, n)[rows] - want) <= 1e-6 * np.linalg.norm(want)

    first = lc.MatMulResidentSession(n, n, n)
    first.start_into(a, b)
    check(first.finish_into())
    q, k, v = (rng.standard_normal((1, 64, 4096, 64), dtype=np.float32) for _ in range(3))
    attn = lc.AttentionSession.batched(1, 64, 4096, 64, compute_dtype="f32")
    o1, o2 = np.empty(q.size, np.float32), np.empty(q.size, np.float32)
    attn.forward_with_policy_into(q, k, v, o1, lc.AttentionIoPolicy())
    resident = lc.AttentionIoPolicy(upload_q=False, upload_k=False, upload_v=False)
    # the second session's operands, product and staging take 1024 MiB; the
    # planes of the first two, 768 and 288 MiB
    with only(hip, 640 * MIB):
        note("[case] second session with 640 MiB left")
        second = lc.MatMulResidentSession(n, n, n)
        second.start_into(a, b)
        check(second.finish_into())
        note("[case] the first sessions without their planes")
        check(first.finish_into())
        attn.forward_with_policy_into(q, k, v, o2, resident)
        assert np.linalg.norm(o2 - o1) <= 2e-6 * np.linalg.norm(o1)
        second.close()
        note("[case] a device buffer of 1200 MiB where 928 are left beside the first session's new planes")
        check(first.finish_into())
        ptr = ctypes.c_void_p()
        assert lc._core._lib().lcMalloc(ctypes.byref(ptr), ctypes.c_size_t(1200 * MIB)) == 0
        assert lc._core._lib().lcFree(ptr) == 0
    note("[case] memory is back")
    check(first.finish_into())
    attn.forward_with_policy_into(q, k, v, o2, lc.AttentionIoPolicy())
    assert np.array_equal(o1, o2)
    first.close()
    attn.close()
