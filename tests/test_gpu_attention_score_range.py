"""Attention whose scores spread widely: the softmax reference is the maximum over
all keys of a tile, whichever lanes hold them.  A reference that misses some lanes'
keys shows as infinities and NaN once a score exceeds it by the type's range.
"""
import numpy as np
import pytest

from gpu_util import require_hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lc():
    return require_hip()


def _round(x, dtype):
    if dtype == "f16":
        return x.astype(np.float16).astype(np.float64)
    if dtype == "bf16":
        u = x.view(np.uint32)
        return ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).astype(np.uint32).view(np.float32).astype(np.float64)
    return x.astype(np.float64)


def _forward(lc, q, k, v, causal, dtype):
    sess = lc.AttentionSession.batched(*q.shape, causal=causal, compute_dtype=dtype)
    out = np.empty(q.size, np.float32)
    sess.forward_with_policy_into(q, k, v, out, lc.AttentionIoPolicy())
    sess.run_cached(2)
    again = np.empty_like(out)
    sess.forward_with_policy_into(q, k, v, again, lc.AttentionIoPolicy(upload_q=False, upload_k=False,
                                                                       upload_v=False))
    sess.close()
    assert np.array_equal(out, again)
    return out.reshape(q.shape)


# (heads, S, D): 16 bits: two and four waves a block, 128-query blocks; fp32: the
# planes kernel with one and two key groups, with and without key splits
@pytest.mark.parametrize("h,s,d", [(2, 200, 64), (1, 64, 128), (40, 130, 128), (64, 96, 64), (9, 520, 64)])
@pytest.mark.parametrize("dtype,peak", [("f16", 30.0), ("bf16", 130.0), ("f32", 130.0)])
@pytest.mark.parametrize("key", [0, 5, 9, 14, 18, 25, 31, 36, 43, 50, 61])
def test_one_key_far_above_the_others(lc, h, s, d, dtype, peak, key):
    """Every other weight is below 2^-43 (a score of 30 in exponent units): the
    output is that key's V, to the last bit of fp32."""
    q = np.zeros((1, h, s, d), np.float32)
    k = np.zeros_like(q)
    v = np.random.default_rng(key).standard_normal(q.shape, dtype=np.float32)
    q[..., 0] = np.sqrt(np.float32(d))
    k[:, :, key, 0] = peak
    got = _forward(lc, q, k, v, False, dtype)
    want = np.broadcast_to(_round(v, dtype)[:, :, key:key + 1], got.shape)
    assert np.abs(got - want).max() <= 2.0 ** -20 * np.abs(want).max()


@pytest.mark.parametrize("h,s,d", [(2, 200, 64), (3, 255, 128), (40, 130, 128), (9, 520, 64)])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype,scale", [("f16", 20.0), ("bf16", 20.0), ("bf16", 60.0), ("f32", 20.0), ("f32", 60.0)])
def test_wide_scores(lc, h, s, d, causal, dtype, scale):
    """Scores of standard deviation `scale`.  With Q and K rounded alike, a score of
    up to 6 deviations carries the rounding of Q times log2(e) (half an ulp of the
    type, averaged over d random terms: 2^-9 or 2^-12 of a deviation; 2^-24 per score
    in fp32) into the exponent; three times that bounds the relative error."""
    rng = np.random.default_rng(5)
    q, k, v = (rng.standard_normal((1, h, s, d), dtype=np.float32) for _ in range(3))
    q *= np.float32(scale)
    got = _forward(lc, q, k, v, causal, dtype)
    rq, rk, rv = (_round(x, dtype) for x in (q, k, v))
    sc = rq @ rk.swapaxes(-1, -2) / np.sqrt(d)
    if causal:
        sc = np.where(np.triu(np.ones((s, s), bool), 1), -np.inf, sc)
    p = np.exp(sc - sc.max(-1, keepdims=True))
    want = (p / p.sum(-1, keepdims=True)) @ rv
    assert np.isfinite(got).all()
    step = {"f16": 2.0 ** -12, "bf16": 2.0 ** -9, "f32": 6 * 2.0 ** -24}[dtype]
    assert np.linalg.norm(got - want) <= 3 * step * scale * np.linalg.norm(want)
