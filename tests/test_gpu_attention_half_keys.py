"""The 16-bit attention that shares a 32-query block's keys between waves
(csrc/kernels/attention.hip, attn_fwd_half_keys_kernel): four waves for few
blocks, two for more.  Sizes where it can go wrong: one query, one past a block
or a key tile, fewer tiles than waves, one tile more than a round of the waves,
batches on both sides of the lines between two and four waves and the
128-query kernel.

Reference: float64 on the rounded operands.  With eps the rounding of the
16-bit type, Q is rounded once more after the scale, which moves a score by at
most delta = eps * scale * sum |q||k|, and every probability is rounded once
(numerator and denominator): |error| <= (e^(2 delta) - 1 + 2 eps) (P |V|), and
2^-16 of it for the fp32 sums.
"""
import numpy as np
import pytest

from gpu_util import require_hip

pytestmark = pytest.mark.gpu

EPS = {"bf16": 2.0**-8, "f16": 2.0**-11}
FEW = [(1, 1, 1, 64), (1, 1, 31, 128), (1, 2, 32, 64), (1, 1, 33, 128), (2, 1, 64, 64), (1, 3, 65, 64), (1, 1, 129, 128),
       (1, 2, 256, 64), (1, 2, 257, 128), (1, 1, 321, 64), (2, 2, 700, 128), (1, 1, 1025, 64)]
# one or two query blocks of at most 32 queries: two waves only where there are many
SHORT = [(20, 20, 1, 128), (10, 40, 31, 128), (30, 20, 32, 64), (25, 20, 17, 64), (25, 20, 33, 64)]
MORE = [(5, 5, 700, 64), (1, 14, 700, 128), (17, 10, 160, 64), (5, 8, 350, 64), (5, 10, 250, 64), (3, 10, 300, 128), (10, 10, 65, 128), (4, 16, 200, 128), (3, 11, 513, 128)]


@pytest.fixture(scope="module")
def lc():
    return require_hip()


def rounded(x, dtype):
    if dtype == "f16":
        return x.astype(np.float16).astype(np.float64)
    u = x.view(np.uint32)
    u = (u + 0x7FFF + ((u >> 16) & 1)) & np.uint32(0xFFFF0000)
    return u.view(np.float32).astype(np.float64)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("shape", FEW + SHORT + MORE, ids=lambda s: "x".join(map(str, s)))
def test_against_float64(lc, shape, dtype, causal):
    b, h, s, d = shape
    rng = np.random.default_rng(s + d)
    q, k, v = (rng.standard_normal((b * h, s, d), dtype=np.float32) for _ in range(3))
    session = lc.AttentionSession.batched(b, h, s, d, causal=causal, compute_dtype=dtype)
    out = np.empty(b * h * s * d, np.float32)
    session.forward_with_policy_into(q.ravel(), k.ravel(), v.ravel(), out, lc.AttentionIoPolicy())
    session.close()
    out = out.reshape(b * h, s, d)
    eps = EPS[dtype]
    mask = np.triu(np.ones((s, s), bool), 1) if causal else np.zeros((s, s), bool)
    for i in range(0, b * h, max(1, b * h // 4)):
        qi, ki, vi = (rounded(x[i], dtype) for x in (q, k, v))
        score = np.where(mask, -np.inf, qi @ ki.T * d**-0.5)
        p = np.exp(score - score.max(axis=1, keepdims=True))
        p /= p.sum(axis=1, keepdims=True)
        delta = eps * d**-0.5 * (np.abs(qi) @ np.abs(ki).T).max(axis=1, keepdims=True)
        bound = (np.expm1(2 * delta) + 2 * eps + 2.0**-16) * (p @ np.abs(vi))
        assert (np.abs(out[i] - p @ vi) <= bound).all()


# four waves, two, 128-query blocks
@pytest.mark.parametrize("heads,s", [(2, 350), (25, 700), (40, 350), (100, 350)])
def test_extreme_scores(lc, heads, s):
    """A row with one +inf score is NaN in every column; a row whose scores lie
    hundreds apart takes the largest one's value; a NaN query stays in its row."""
    d = 64
    rng = np.random.default_rng(heads)
    q, k, v = (rng.standard_normal((heads, s, d), dtype=np.float32) for _ in range(3))
    q[0, 5] = 0.0
    q[0, 5, 0] = 3.0e38
    k[0, 40, 0] = 3.0e38
    q[1, 7] = np.nan
    q[1, 9] = 0.0
    q[1, 9, 0] = 8.0
    k[1, :, 0] = np.linspace(-1000.0, 1000.0, s) * (s / 350)
    session = lc.AttentionSession.batched(1, heads, s, d, causal=False, compute_dtype="bf16")
    out = np.empty(heads * s * d, np.float32)
    session.forward_with_policy_into(q.ravel(), k.ravel(), v.ravel(), out, lc.AttentionIoPolicy())
    session.close()
    out = out.reshape(heads, s, d)
    assert np.isnan(out[0, 5]).all()
    assert np.isnan(out[1, 7]).all()
    assert np.isfinite(out[1, 8]).all() and np.isfinite(out[1, 6]).all()
    # the last key leads the next by more than 5 in the exponent
    assert np.allclose(out[1, 9], v[1, -1], rtol=0.02, atol=0.06)
