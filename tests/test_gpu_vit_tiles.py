"""The ViT block's GEMMs on the tiles of csrc/kernels/gemm_half.hip (16-bit
ReLU rows, the QKV projection to head-major Q / K and transposed V, fp32 rows)
against the register-staged kernels (CJ_HIP_VIT_RING=0).  fp32 sums that differ
in their last bits can move a value that is rounded to 16 bits by one step
(2^-7 of it in bf16, 2^-10 in f16), at three places on the way (tokens, Q / K /
V, attention output), so the 2-norm of the difference stays below three such
steps of the result's; a misplaced element or row is of the result's own size.
Rows from one image's few tokens to several rounds of the
largest tile, tokens per image that are no multiple of 4, 16 or 64, images that
share a row block, heads of 64 and 128, widths with less than a column tile.
"""
import numpy as np
import pytest

from gpu_util import require_hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lc():
    return require_hip()


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("batch,ih,iw,patch,embed,heads", [
    (1, 16, 16, 16, 64, 1),      # one token
    (1, 112, 112, 16, 768, 12),  # 49 rows
    (3, 40, 40, 8, 192, 3),      # 25 tokens an image
    (1, 224, 224, 16, 768, 12),
    (2, 96, 256, 16, 256, 2),    # heads of 128
    (8, 224, 224, 16, 768, 12),
    (17, 224, 224, 16, 768, 12),
    (5, 256, 256, 8, 320, 5),    # 1024 tokens an image
])
def test_agrees_with_the_staged_kernels(lc, monkeypatch, batch, ih, iw, patch, embed, heads, dtype):
    rng = np.random.default_rng(batch * ih + embed)
    x = rng.standard_normal((batch, 3, ih, iw), dtype=np.float32)
    w_conv = rng.standard_normal((embed, 3, patch, patch), dtype=np.float32) * np.float32((3 * patch**2) ** -0.5)
    w_qkv = rng.standard_normal((embed, 3 * embed), dtype=np.float32) * np.float32(embed**-0.5)
    w_o = rng.standard_normal((embed, embed), dtype=np.float32) * np.float32(embed**-0.5)
    tiles = lc.vit_block(x, w_conv, w_qkv, w_o, heads, compute_dtype=dtype)
    monkeypatch.setenv("CJ_HIP_VIT_RING", "0")
    staged = lc.vit_block(x, w_conv, w_qkv, w_o, heads, compute_dtype=dtype)
    assert np.isfinite(tiles).all()
    step = {"bf16": 2.0**-7, "f16": 2.0**-10}[dtype]
    rows = np.linalg.norm((tiles - staged).reshape(-1, embed), axis=1)
    assert (rows <= 3 * step * np.linalg.norm(staged.reshape(-1, embed), axis=1)).all()
