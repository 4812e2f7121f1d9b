"""The fp32 attention forward on bf16 planes (csrc/kernels/attention_f32.hip)
vs float64, where its blocks end: the head dims it takes, sequences around a
32-key tile and a 128-query block, key splits and none, one and two key groups,
causal and not, the postprocess, and operands that three bf16 values cannot
hold (they take the fp32 matrix instruction).

Tolerance: scores and outputs are sums of exact products accumulated in fp32,
so against float64 the relative error (2-norm) stays within 2e-6, four times the
largest this kernel shows over these cases.
"""
import numpy as np
import pytest

from gpu_util import note, require_hip

pytestmark = pytest.mark.gpu

TOL = 2e-6


@pytest.fixture(scope="module")
def lc():
    return require_hip()


def _reference(q, k, v, causal):
    q, k, v = (x.astype(np.float64) for x in (q, k, v))
    with np.errstate(all="ignore"):
        s = q @ np.swapaxes(k, -1, -2) / np.sqrt(q.shape[-1])
        if causal:
            n = s.shape[-1]
            s = np.where(np.arange(n)[None, :] > np.arange(n)[:, None], -1e30, s)
        p = np.exp(s - s.max(-1, keepdims=True))
        return (p / p.sum(-1, keepdims=True)) @ v


def _inputs(shape, seed=3):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal(shape, dtype=np.float32) for _ in range(3)]


# (batch, heads, S, D): more than 256 blocks of 16 queries, so not the 16-query
# kernel at D <= 64; larger head dims always
SHAPES = [(1, 40, 97, 32), (2, 40, 127, 32), (3, 43, 129, 64), (2, 64, 65, 64), (1, 70, 160, 64), (300, 1, 33, 64),
          (1, 9, 1025, 64), (1, 2, 31, 96), (1, 3, 300, 96), (1, 1, 1, 128), (1, 2, 128, 128), (1, 1, 513, 128)]


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,h,s,d", SHAPES)
def test_split_forward_against_float64(lc, b, h, s, d, causal):
    q, k, v = _inputs((b, h, s, d))
    got = lc.attention_batched(q, k, v, causal=causal, compute_dtype="f32").astype(np.float64)
    ref = _reference(q, k, v, causal)
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    note(f"[parity] f32 split attention {(b, h, s, d)} causal={causal}: rel {err:.2e}")
    assert err <= TOL


def test_split_forward_resident_and_postprocess(lc):
    b, h, s, d = 1, 9, 1025, 64
    q, k, v = _inputs((b, h, s, d))
    ref = _reference(q, k, v, True)
    sess = lc.AttentionSession.batched(b, h, s, d, causal=True, compute_dtype="f32")
    out = np.empty(q.size, np.float32)
    sess.forward_with_policy_into(q, k, v, out, lc.AttentionIoPolicy())
    again = np.empty_like(out)
    sess.run_cached(3)
    resident = dict(upload_q=False, upload_k=False, upload_v=False)
    sess.forward_with_policy_into(q, k, v, again, lc.AttentionIoPolicy(**resident))
    assert np.array_equal(out, again)
    post = np.empty_like(out)
    sess.forward_with_policy_into(q, k, v, post, lc.AttentionIoPolicy(output_scale=1.5, output_bias=-0.25,
                                                                       output_relu=True, **resident))
    want = np.maximum(ref * 1.5 - 0.25, 0.0).ravel()
    assert np.linalg.norm(post - want) <= TOL * np.linalg.norm(want)
    # one tensor replaced, the others resident
    v2 = _inputs((b, h, s, d), seed=5)[0]
    sess.forward_with_policy_into(q, k, v2, out, lc.AttentionIoPolicy(upload_q=False, upload_k=False))
    want = _reference(q, k, v2, True).ravel()
    assert np.linalg.norm(out - want) <= TOL * np.linalg.norm(want)
    sess.close()


@pytest.mark.parametrize("b,h,s,d", [(1, 9, 520, 64), (1, 2, 200, 128), (2, 40, 127, 32), (1, 3, 300, 96)])
@pytest.mark.parametrize("what", ["nan", "inf", "tiny", "huge"])
def test_operands_outside_the_split(lc, b, h, s, d, what):
    q, k, v = _inputs((b, h, s, d))
    if what == "nan":
        v[0, 0, 5, 7] = np.nan
    elif what == "inf":
        v[0, h - 1, s - 1, 0] = np.inf
    elif what == "tiny":
        q *= np.float32(1e-33)
        k *= np.float32(1e33)
    else:
        v *= np.float32(1e30)
    causal = what in ("tiny", "huge")  # non-finite values and masks: the next test
    ref = _reference(q, k, v, causal)
    sess = lc.AttentionSession.batched(b, h, s, d, causal=causal, compute_dtype="f32")
    first, later = np.empty(q.size, np.float32), np.empty(q.size, np.float32)
    sess.forward_with_policy_into(q, k, v, first, lc.AttentionIoPolicy())  # the kernel's own check may decide
    sess.forward_with_policy_into(q, k, v, later, lc.AttentionIoPolicy(upload_q=False, upload_k=False,
                                                                       upload_v=False))  # the host knows
    sess.close()
    fine = np.isfinite(ref.ravel())
    for got in (first, later):
        np.testing.assert_array_equal(np.where(fine, 0.0, got), np.where(fine, 0.0, ref.ravel()))
        assert np.all(np.isfinite(got[fine]))
        assert np.linalg.norm(got[fine] - ref.ravel()[fine]) <= TOL * np.linalg.norm(ref.ravel()[fine])


# (heads, S, D): two key groups with and without key splits, one group (D = 128)
# with and without, enough blocks for none of either
@pytest.mark.parametrize("h,s,d", [(9, 520, 64), (9, 1025, 64), (70, 160, 64), (2, 200, 128), (1, 600, 128),
                                   (40, 300, 128)])
@pytest.mark.parametrize("what", ["nan", "inf"])
@pytest.mark.parametrize("key", [33, 100, 127])
def test_causal_non_finite_value_stays_behind_its_tile(lc, h, s, d, what, key):
    """A non-finite V row meets a masked query as 0 * inf only within the query's
    own 32 keys: every earlier row is finite, whether the kernel finds the value
    (first call) or the host has seen it (later calls)."""
    q, k, v = _inputs((1, h, s, d))
    ref = _reference(q, k, v, True)[0]
    v[0, 0, key, 3] = np.nan if what == "nan" else np.inf
    sess = lc.AttentionSession.batched(1, h, s, d, causal=True, compute_dtype="f32")
    first, later = np.empty(q.size, np.float32), np.empty(q.size, np.float32)
    sess.forward_with_policy_into(q, k, v, first, lc.AttentionIoPolicy())
    sess.forward_with_policy_into(q, k, v, later, lc.AttentionIoPolicy(upload_q=False, upload_k=False,
                                                                       upload_v=False))
    sess.close()
    assert np.array_equal(np.isfinite(first), np.isfinite(later))
    tile = key // 32 * 32
    for got in (first.reshape(h, s, d), later.reshape(h, s, d)):
        assert not np.isfinite(got[0, key:, 3]).any()  # a query that sees the value
        got[0, tile:, 3] = ref[0, tile:, 3]
        assert np.isfinite(got).all()
        assert np.linalg.norm(got - ref) <= TOL * np.linalg.norm(ref)
