"""The fp32 GEMM on bf16 planes (csrc/kernels/gemm_f32.hip) vs float64.

Every variant is forced through a seeded tune cache at the sizes where its
tiles, its k steps or its split of k end: one row or column, one below and one
above a tile, one k step, fewer steps than waves, more steps than the LDS ring
has slots, several workgroups a tile.  Bound per element: every output is a sum
of K exact products; each accumulation rounds (or truncates) to at most 2^-23
of the running sum of magnitudes, and a value passes through at most
6 K / 32 + 16 of them, so |error| <= (6 K / 32 + 16) * 2^-23 * (|A| |B|).

Operands that three bf16 values cannot hold exactly (infinities, NaN, tiny and
huge values) take the fp32 matrix instruction and must give what it gives.
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
VARIANTS = {"f32_split_64x64": "64,64,32,4,4", "f32_split_80x64": "80,64,32,4,4",
            "f32_split_128x128": "128,128,32,4,1"}
SHAPES = [(1, 1, 1), (1, 300, 65), (63, 33, 64), (64, 32, 63), (65, 64, 129), (81, 97, 64), (127, 160, 128),
          (129, 225, 127), (160, 512, 257), (300, 3000, 300), (257, 1056, 513)]


@pytest.fixture(scope="module")
def lc():
    return require_hip()


def _child(code, cwd):
    env = dict(os.environ, PYTHONPATH=os.path.join(ROOT, "lightining-core_amd"))
    r = subprocess.run([sys.executable, "-u", "-c", textwrap.dedent(code)], cwd=cwd, env=env, capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


@pytest.mark.parametrize("name", sorted(VARIANTS))
def test_split_variants_against_float64(lc, tmp_path, name):
    cache = tmp_path / "mm.csv"
    cache.write_text("#lc_tune_cache,matmul,2\n" +
                     "".join(f"{m},{k},{n},0,gfx950,{name},{VARIANTS[name]}\n" for m, k, n in SHAPES))
    out = _child(f"""
        import numpy as np
        import lightning_core as lc
        from lightning_core import synth
        lc.tune_cache_load({str(cache)!r})
        for m, k, n in {SHAPES!r}:
            print("[case]", m, k, n, flush=True)
            a, b = synth.normal((m, k), stream=41), synth.normal((k, n), stream=42)
            s = lc.MatMulResidentSession(m, k, n)
            assert s.start_into(a, b) is not None and {name!r} in s.kernel_name()
            c = s.finish_into().reshape(m, n)
            again = s.finish_into().reshape(m, n)
            s.close()
            assert np.array_equal(c, again)
            a, b = a.astype(np.float64), b.astype(np.float64)
            bound = (6 * k / 32 + 16) * 2.0 ** -23 * (np.abs(a) @ np.abs(b))
            print("WORST", m, k, n, float((np.abs(c - a @ b) / bound).max()), flush=True)
    """, tmp_path)
    worst = [line.split()[1:] for line in out.splitlines() if line.startswith("WORST")]
    assert len(worst) == len(SHAPES)
    for m, k, n, share in worst:
        note(f"[parity] {name} {m}x{k}x{n}: {float(share):.3f} of the bound")
        assert float(share) <= 1.0


@pytest.mark.parametrize("m,k,n", [(70, 96, 130), (200, 512, 300), (2048, 1024, 2048)])
@pytest.mark.parametrize("what", ["nan", "inf", "tiny", "huge", "lowest", "zero"])
def test_operands_outside_the_split(lc, m, k, n, what):
    rng = np.random.default_rng(7)
    a = rng.standard_normal((m, k), dtype=np.float32)
    b = rng.standard_normal((k, n), dtype=np.float32)
    if what == "nan":
        a[m // 2, k // 3] = np.nan
    elif what == "inf":
        b[k // 3, n // 2] = -np.inf
    elif what == "tiny":  # below 2^-100, where a low part would leave bf16's range
        a *= np.float32(1e-34)
        b *= np.float32(1e30)
    elif what == "huge":
        a *= np.float32(1e19)
        b *= np.float32(1e15)
    elif what == "lowest":
        a[0] = 0.0
        a[0, k // 2] = np.finfo(np.float32).min  # one product a row: no partial sum overflows on the way
    else:
        a[:] = 0.0
    with np.errstate(all="ignore"):
        a64, b64 = a.astype(np.float64), b.astype(np.float64)
        ref = a64 @ b64
        bound = (k + 16) * 2.0 ** -23 * (np.abs(a64) @ np.abs(b64))
    s = lc.matmul2d_resident_session(a, b)
    out = s.start_into(a, b)
    first = s.finish_into(out=out).copy().reshape(m, n)  # the kernel's own check may still decide
    lc.device_synchronize()
    later = s.finish_into(out=out).reshape(m, n)  # the host knows
    s.close()
    call = lc.matmul2d(a, b)
    clear = np.isfinite(ref) & (np.abs(ref) + bound < 3.0e38)
    with np.errstate(all="ignore"):
        special = np.where(clear, 0.0, ref.astype(np.float32))
    for got in (first, later, call):
        edge = ~clear & np.isfinite(ref) & (np.abs(ref) <= np.finfo(np.float32).max + bound)  # may round either way
        np.testing.assert_array_equal(np.where(clear | edge, 0.0, got), np.where(edge, 0.0, special))
        assert np.all(np.isfinite(got[clear]))
        assert np.all(np.abs(got[clear] - ref[clear]) <= bound[clear])


def test_guard_follows_each_upload(lc):
    # A fit operand after an unfit one, and back, on one session.
    rng = np.random.default_rng(9)
    m, k, n = 130, 200, 70
    a = rng.standard_normal((m, k), dtype=np.float32)
    b = rng.standard_normal((k, n), dtype=np.float32)
    bad = a.copy()
    bad[3, 5] = np.inf
    s = lc.MatMulResidentSession(m, k, n)
    for x in (a, bad, a, bad, bad, a):
        s.start_into(x, b)
        got = s.finish_into().reshape(m, n)
        with np.errstate(all="ignore"):
            ref = x.astype(np.float64) @ b.astype(np.float64)
        fin = np.isfinite(ref)
        assert np.array_equal(fin, np.isfinite(got)) and np.array_equal(got[~fin], ref[~fin].astype(np.float32))
        assert np.abs(got[fin] - ref[fin]).max() <= 1e-5 * np.abs(ref[fin]).max()
    s.close()


def test_plain_calls_do_not_depend_on_what_ran_before(lc, tmp_path):
    """Equal matmul2d calls give equal bits: the first of a shape, a later one,
    one after a resident session has timed the split variants, and one in a
    process that finds the tune cache of the first; below 2^32 products none of
    them runs a split variant, and the session still does where it is faster."""
    shapes = [(600, 700, 500), (640, 2048, 640), (1000, 777, 1030), (64, 64, 64)]
    body = f"""
        import hashlib
        import sys
        import lightning_core as lc
        from lightning_core import synth
        for m, k, n in {shapes!r}:
            print("[case]", m, k, n, flush=True)
            a, b = synth.normal((m, k), stream=61), synth.normal((k, n), stream=62)
            calls = [lc.matmul2d(a, b) for _ in range(3)]
            s = lc.MatMulResidentSession(m, k, n)
            s.start_into(a, b)
            s.finish_into()
            name = s.kernel_name()
            s.close()
            calls.append(lc.matmul2d(a, b))
            print("SHA", m, k, n, name.split()[0], *(hashlib.sha256(c.tobytes()).hexdigest() for c in calls), flush=True)
    """
    rows = [[line.split()[1:] for line in _child(body, tmp_path).splitlines() if line.startswith("SHA")]
            for _ in range(2)]
    cached = [r.split(",") for r in (tmp_path / ".lightning_core_matmul_tune_cache.csv").read_text().splitlines()
              if not r.startswith("#")]
    assert len(rows[0]) == len(shapes) == len(cached)
    for first, again in zip(*rows):
        assert len(set(first[4:] + again[4:])) == 1, first[:3]
        assert first[3] == again[3]  # the session's variant comes from the cache
        once, _, resident = next(r[5] for r in cached if r[:3] == first[:3]).partition("|")
        assert "split" not in once and (resident or once) == first[3]
    assert any("split" in r[3] for r in rows[0])


def test_unfit_operands_settle_no_split_choice(lc, tmp_path):
    """The choice of a resident launch's variant is timed on operands the split
    GEMM takes: a session that starts with one it does not take leaves it open,
    in the session and in the tune cache, and the next fit upload settles it."""
    cache = tmp_path / ".lightning_core_matmul_tune_cache.csv"
    out = _child(f"""
        import numpy as np
        import lightning_core as lc
        from lightning_core import synth
        def row():
            return next(r.split(",")[5] for r in open({str(cache)!r}) if r.startswith("640,2048,640,"))
        m, k, n = 640, 2048, 640
        a, b = synth.normal((m, k), stream=71), synth.normal((k, n), stream=72)
        bad = a.copy()
        bad[1, 2] = 1e-35
        s = lc.MatMulResidentSession(m, k, n)
        for _ in range(2):
            s.start_into(bad, b)
            c = s.finish_into().reshape(m, n)
            assert np.abs(c - bad.astype(np.float64) @ b).max() <= 1e-4 * np.abs(c).max()
            print("ROW", row(), flush=True)
        s.start_into(a, b)
        s.finish_into()
        print("ROW", row(), s.kernel_name().split()[0], flush=True)
        s.close()
    """, tmp_path)
    rows = [line.split()[1:] for line in out.splitlines() if line.startswith("ROW")]
    for (name,) in rows[:2]:
        once, bar, resident = name.partition("|")
        assert bar and not resident and "split" not in once
    name, kernel = rows[2]
    assert name.partition("|")[2] == kernel and "split" in kernel


def test_kernel_name_follows_the_operands(lc):
    """kernel_name() is the GEMM that runs: with operands the split GEMM does not
    take it names the fp32 instruction's kernel, and the shape's own again after
    the next fit upload."""
    rng = np.random.default_rng(10)
    m, k, n = 640, 2048, 640
    a = rng.standard_normal((m, k), dtype=np.float32)
    b = rng.standard_normal((k, n), dtype=np.float32)
    bad = a.copy()
    bad[3, 5] = np.inf
    s = lc.MatMulResidentSession(m, k, n)
    names = {True: set(), False: set()}
    for x in (a, bad, a, bad):
        s.start_into(x, b)
        s.finish_into()
        names[x is a].add(s.kernel_name().split()[0])
    s.close()
    assert len(names[True]) == 1 and "split" in names[True].pop()
    assert not any("split" in x for x in names[False])


def test_heuristic_keeps_whole_tiles_for_the_shortest_k(lc, tmp_path):
    """Without autotune: one k step in few tiles, or a few in many tiles with rows
    that no 16-byte store fits, run the fp32 instruction's kernels; the split GEMM
    begins past those lines."""
    shapes = {(948, 45, 631): False, (64, 64, 64): False, (710, 51, 1918): False, (1500, 190, 1501): False,
              (1500, 193, 1501): True, (1024, 32, 2816): True, (1024, 65, 1024): True, (1024, 1024, 1024): True}
    out = _child(f"""
        import os
        os.environ["CJ_MATMUL_AUTOTUNE"] = "0"
        import numpy as np
        import lightning_core as lc
        from lightning_core import synth
        for m, k, n in {list(shapes)!r}:
            a, b = synth.normal((m, k), stream=81), synth.normal((k, n), stream=82)
            s = lc.MatMulResidentSession(m, k, n)
            s.start_into(a, b)
            c = s.finish_into().reshape(m, n)
            print("NAME", m, k, n, s.kernel_name().split()[0], flush=True)
            s.close()
            a, b = a.astype(np.float64), b.astype(np.float64)
            bound = (k + 16) * 2.0 ** -23 * (np.abs(a) @ np.abs(b))
            assert (np.abs(c - a @ b) <= bound).all()
    """, tmp_path)
    names = [line.split()[1:] for line in out.splitlines() if line.startswith("NAME")]
    assert [("split" in name) for *_, name in names] == list(shapes.values())


def _exact64(x):
    """fp32 to fp64 bit by bit: a library built with -ffast-math may have set this
    process to read subnormal values as zeros."""
    u = x.view(np.uint32)
    exponent = ((u >> 23) & 255).astype(np.int64)
    mantissa = (u & 0x7FFFFF).astype(np.float64) + np.where(exponent > 0, 2.0 ** 23, 0.0)
    return np.where(u >> 31, -1.0, 1.0) * np.ldexp(mantissa, np.maximum(exponent, 1) - 150)


@pytest.mark.parametrize("e", [-50, -59, -62, -66])
@pytest.mark.parametrize("m,k,n", [(256, 256, 256), (300, 512, 1024), (2048, 256, 2048)])
def test_products_in_the_subnormal_range(lc, m, k, n, e):
    """Operands near 2^e fit the planes, and their small products lie below 2^-126
    from e = -55 on: they count in full (a sum below 2^-126 keeps steps of 2^-149),
    where flushing them to zero would cost 2^-8 of the result."""
    rng = np.random.default_rng(11)
    scale = np.float32(2.0) ** np.float32(e)
    a = rng.standard_normal((m, k), dtype=np.float32) * scale
    b = rng.standard_normal((k, n), dtype=np.float32) * scale
    s = lc.MatMulResidentSession(m, k, n)
    s.start_into(a, b)
    got = _exact64(s.finish_into()).reshape(m, n)
    assert "split" in s.kernel_name()
    s.close()
    a, b = a.astype(np.float64), b.astype(np.float64)
    bound = (6 * k / 32 + 16) * 2.0 ** -23 * (np.abs(a) @ np.abs(b)) + (6 * k + 16) * 2.0 ** -149
    assert (np.abs(got - a @ b) <= bound).all()
