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


# More than 64 tiles of 128 x 128, few k steps or columns that no 16-byte store fits: the
# register-staged kernels take about half of the ring tiles' time there.
STORES = [(7044, 157, 1759), (3030, 91, 2554), (2034, 260, 6795)]
# Long k: the ring tiles take about half of the others' time.
LONG = [(1500, 3000, 2000), (378, 7510, 2692)]


@pytest.mark.parametrize("tuned", ["1", "0"])
def test_products_that_are_mostly_stores_keep_the_staged_kernels(lc, tmp_path, tuned):
    """Both the timed choice and the heuristic's; results against float64 as above."""
    env = dict(os.environ, PYTHONPATH=os.path.join(ROOT, "lightining-core_amd"), CJ_MATMUL_AUTOTUNE=tuned)
    r = subprocess.run([sys.executable, "-u", "-c", textwrap.dedent(f"""
        import numpy as np
        import lightning_core as lc
        from lightning_core import synth
        for m, k, n in {STORES + LONG!r}:
            print("[case]", m, k, n, flush=True)
            a, b = synth.normal((m, k), stream=53), synth.normal((k, n), stream=54)
            s = lc.MatMulResidentSession(m, k, n, compute_dtype="bf16")
            s.start_into(a, b)
            name = s.kernel_name().split()[0]
            c = s.finish_into().reshape(m, n)[-130:]
            s.close()
            a, b = (synth.round_to(x, "bf16").astype(np.float64) for x in (a[-130:], b))
            bound = (k / 32 + 8) * 2.0 ** -22 * (np.abs(a) @ np.abs(b))
            print("NAME", m, k, n, name, float((np.abs(c - a @ b) / bound).max()), flush=True)
    """)], cwd=tmp_path, env=env, capture_output=True, text=True, timeout=110)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    names = [line.split()[1:] for line in r.stdout.splitlines() if line.startswith("NAME")]
    assert len(names) == len(STORES + LONG)
    for m, k, n, name, share in names:
        note(f"[tune] {m}x{k}x{n}: {name}, {float(share):.3f} of the bound")
        assert float(share) <= 1.0
        assert ("_r4_" in name) == ((int(m), int(k), int(n)) in LONG)
