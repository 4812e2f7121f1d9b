"""The 16-bit GEMM tiles of csrc/kernels/gemm_half.hip, each forced through a
seeded tune cache where its tiles and its ring of four stages end: fewer rows
than a tile, one row or column past it, rows of tiles that reach past the padded
operand, one stage, three to six stages.

Every accumulator adds its k steps in the order of the 256x256 kernel, so the
results must equal that kernel's bit for bit; that kernel's are held against
float64: |error| <= (K / 32 + 8) * 2^-22 * (|A| |B|) on the rounded operands (a
step adds 32 exact products with at most one truncation of the sum).
"""
import os
import subprocess
import sys
import textwrap

import numpy as np
import pytest

from gpu_util import note, require_hip

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BASE = ("half_w4h_256x256", "256,256,64,4,1")
TILES = [("half_r4_128x128", "128,128,64,4,1"), ("half_r4_96x128", "96,128,64,4,1"),
         ("half_r4_64x128", "64,128,64,4,1"), ("half_r4_64x64", "64,64,64,4,1"), ("half_r4_32x64", "32,64,64,4,1")]
SHAPES = [(17, 64, 1), (31, 50, 65), (33, 128, 129), (65, 190, 64), (96, 256, 128), (97, 320, 127), (129, 384, 257),
          (500, 1000, 300), (1024, 192, 700)]


@pytest.fixture(scope="module")
def lc():
    return require_hip()


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_tiles_match_the_256_tile_bitwise(lc, tmp_path, dtype):
    code = {"bf16": 1, "f16": 2}[dtype]
    caches = []
    for name, cols in [BASE] + TILES:
        cache = tmp_path / f"{name}.csv"
        cache.write_text("#lc_tune_cache,matmul,2\n" +
                         "".join(f"{m},{k},{n},{code},gfx950,{name},{cols}\n" for m, k, n in SHAPES))
        caches.append((name, str(cache)))
    env = dict(os.environ, PYTHONPATH=os.path.join(ROOT, "lightining-core_amd"))
    r = subprocess.run([sys.executable, "-u", "-c", textwrap.dedent(f"""
        import numpy as np
        import lightning_core as lc
        from lightning_core import synth
        base = {{}}
        for name, cache in {caches!r}:
            lc.tune_cache_load(cache)
            for m, k, n in {SHAPES!r}:
                print("[case]", name, m, k, n, flush=True)
                a, b = synth.normal((m, k), stream=51), synth.normal((k, n), stream=52)
                s = lc.MatMulResidentSession(m, k, n, compute_dtype={dtype!r})
                s.start_into(a, b)
                assert name in s.kernel_name(), s.kernel_name()
                c = s.finish_into().reshape(m, n)
                s.close()
                if name == {BASE[0]!r}:
                    base[m, k, n] = c
                    a, b = (synth.round_to(x, {dtype!r}).astype(np.float64) for x in (a, b))
                    bound = (k / 32 + 8) * 2.0 ** -22 * (np.abs(a) @ np.abs(b))
                    print("WORST", m, k, n, float((np.abs(c - a @ b) / bound).max()), flush=True)
                else:
                    assert np.array_equal(c, base[m, k, n]), (name, m, k, n)
    """)], cwd=tmp_path, env=env, capture_output=True, text=True, timeout=110)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    worst = [line.split()[1:] for line in r.stdout.splitlines() if line.startswith("WORST")]
    assert len(worst) == len(SHAPES)
    for m, k, n, share in worst:
        note(f"[parity] {dtype} {m}x{k}x{n}: {float(share):.3f} of the bound")
        assert float(share) <= 1.0
