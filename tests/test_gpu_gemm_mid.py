"""GPU: the medium-tile W8A8 GEMM at the edges of its tiles, K stages, scale chunks and K
splits, for every recipe, against the fp64 product of the same operands under the
package's stated tolerance (``tests/_tol.py``); INT8 against the exact integer sum."""

import pytest
import torch

from tests._tol import assert_linear_close

pytestmark = pytest.mark.gpu
FP8 = torch.float8_e4m3fn


def _fp8(shape, g):
    return (torch.randn(shape, generator=g, device=g.device) * 50).clamp(-448, 448).to(FP8)


def _expand(scale, rows, cols, by, bx):
    return scale.double().repeat_interleave(by, 0)[:rows].repeat_interleave(bx, 1)[:, :cols]


def _wide(t, stride, dev):
    """``t`` on the device, its rows ``stride`` elements apart (None: contiguous)."""
    t = t.to(dev)
    if stride is None:
        return t
    rows = torch.empty((t.shape[0] - 1) * stride + t.shape[1], dtype=torch.uint8, device=dev).view(t.dtype)
    view = rows.as_strided(t.shape, (stride, 1))
    view.copy_(t)
    return view


def _run(recipe, m, n, k, bias, odt, col_major, gpu, lda=None, ldw=None, on="cpu", pad=0):
    """(output, fp64 reference, plan) of one call with seeded operands, drawn on device ``on``;
    ``pad`` columns behind the output's stay as they were."""
    from ayaka.kernel.hip import _lib, fp8_blockwise_mm, fp8_scaled_mm, int8_scaled_mm, mxfp8_scaled_mm

    g = torch.Generator(device=on).manual_seed(m * 131 + n * 7 + k)
    draw = lambda *shape: torch.rand(*shape, generator=g, device=on)  # noqa: E731
    if recipe == "int8":
        a, w = (torch.randint(-127, 128, (r, k), generator=g, dtype=torch.int8, device=on) for r in (m, n))
    else:
        a, w = _fp8((m, k), g), _fp8((n, k), g)
    ag, wg = _wide(a, lda, gpu), _wide(w, ldw, gpu)
    b = torch.randn(n, generator=g, device=on).to(odt) if bias else None
    buffer = torch.full((m, n + pad), 7.0, dtype=odt, device=gpu)
    out = buffer[:, :n]
    bg = None if b is None else b.to(gpu)
    if recipe == "int8":
        int8_scaled_mm(ag, wg.t(), torch.ones(m, device=gpu), torch.ones(n, device=gpu), bias=bg, out=out)
        sa = sb = 1.0
    elif recipe == "scaled":
        sa, sb = draw(m) * 1e-2, draw(n) * 1e-2
        fp8_scaled_mm(ag, wg.t(), sa.to(gpu), sb.to(gpu), bias=bg, out=out)
        sa, sb = sa[:, None].double(), sb[:, None].double()
    elif recipe == "scalar":
        sa, sb = torch.tensor(0.003), torch.tensor(0.02)
        fp8_scaled_mm(ag, wg.t(), sa.to(gpu), sb.to(gpu), bias=bg, out=out)
    elif recipe in ("block", "block16"):
        kb = -(-k // 128)
        ta, tb = draw(m, kb) * 1e-2, draw(-(-n // 128), kb) * 1e-2
        if not col_major:
            tb = tb.to(torch.bfloat16)
        if recipe == "block16":
            ta = ta.to(torch.float16)
        table = ta.t().contiguous() if col_major else ta
        fp8_blockwise_mm(ag, wg, table.to(gpu), tb.to(gpu), bias=bg, out=out, a_scale_col_major=col_major)
        sa, sb = _expand(ta, m, k, 1, 128), _expand(tb, n, k, 128, 128)
    else:
        ca, cb = (torch.randint(112, 122, (r, k // 32), generator=g, dtype=torch.uint8, device=on) for r in (m, n))
        mxfp8_scaled_mm(ag, ca.to(gpu), wg, cb.to(gpu), bg, out=out)
        sa, sb = (_expand(torch.exp2(c.double() - 127), c.shape[0], k, 1, 32) for c in (ca, cb))
    plan = _lib.last_plan()
    assert (buffer[:, n:] == 7).all(), "wrote past the output columns"
    ref = (a.double() * sa).to(gpu) @ (w.double() * sb).to(gpu).t()
    return out, ref if b is None else ref + bg.double(), plan


@pytest.mark.parametrize("recipe,m,n,k,bias,odt,col_major", [  # most on 64 x 64 tiles
    ("scaled", 65, 129, 16, True, torch.float32, False),       # one short stage
    ("scaled", 100, 128, 128, False, torch.bfloat16, False),   # exact stage
    ("scaled", 33, 1001, 4112, True, torch.float16, False),    # K tail, odd N, split
    ("scaled", 300, 2052, 3696, True, torch.float16, False),   # K % 64 != 0
    ("scalar", 255, 300, 2064, False, torch.float32, False),   # odd stage count
    ("scaled", 1025, 3072, 1024, True, torch.bfloat16, False),
    ("scaled", 700, 9000, 2096, False, torch.bfloat16, False),
    ("block", 70, 130, 128, True, torch.bfloat16, True),
    ("block", 65, 1000, 4096, False, torch.float16, True),     # split
    ("block", 129, 2052, 1152, True, torch.float32, False),    # row-major, bf16 weight scales
    ("block", 40, 100, 384, False, torch.bfloat16, False),     # N < 128
    ("block", 1000, 4096, 4096, False, torch.bfloat16, True),
    ("mx", 66, 136, 512, True, torch.float32, False),          # one code chunk
    ("mx", 100, 1000, 4096, False, torch.bfloat16, False),     # split in whole chunks
    ("mx", 70, 260, 1184, True, torch.float16, False),         # K % 128 != 0: unaligned codes
    ("mx", 40, 300, 2688, False, torch.bfloat16, False),       # K % 512 != 0
    ("mx", 200, 2050, 2944, True, torch.float32, False),       # K % 512 != 0, several tiles a side
    ("mx", 40, 4096, 11008, False, torch.bfloat16, False),     # a K the decode kernel cannot split
    ("mx", 300, 3072, 1536, True, torch.bfloat16, False),
])
def test_medium_tiles(gpu, recipe, m, n, k, bias, odt, col_major):
    print(f"medium tiles recipe={recipe} m={m} n={n} k={k} bias={bias} out={odt} col_major={col_major}", flush=True)
    out, ref, plan = _run(recipe, m, n, k, bias, odt, col_major, gpu)
    assert plan.startswith("mid "), plan
    assert_linear_close(out, ref, f"{recipe} {m}x{n}x{k}")


@pytest.mark.parametrize("recipe,k", [("scaled", 4096), ("block", 4096), ("mx", 4096), ("mx", 1184)])
@pytest.mark.parametrize("n", [641, 642, 644, 648])
def test_medium_tiles_half_outputs(gpu, recipe, k, n):
    """16-bit outputs are the fp32 output rounded once, whatever part of their rows is aligned
    (16 bytes for N % 8 == 0, 8 for every other row of N % 8 == 4)."""
    m = 97
    full, _, plan = _run(recipe, m, n, k, False, torch.float32, False, gpu)
    for odt in (torch.bfloat16, torch.float16):
        half, _, plan2 = _run(recipe, m, n, k, False, odt, False, gpu)
        assert plan == plan2 and torch.equal(half, full.to(odt))


@pytest.mark.parametrize("recipe", ["scaled", "block", "block16", "mx", "int8"])
@pytest.mark.parametrize("m,k,n,pad", [(70, 256, 16633, 0), (70, 256, 16634, 1), (70, 256, 16635, 5), (70, 384, 16636, 0),
                                       (1030, 256, 1031, 2), (137, 4096, 16634, 0), (137, 4224, 16634, 0)])
def test_medium_tiles_large_f32_outputs(gpu, recipe, m, k, n, pad):
    """fp32 outputs of 2^20 elements and more, which pass through LDS up to K = 4096: rows of every
    alignment, and the 16-bit outputs are their rounding."""
    print(f"large fp32 output recipe={recipe} m={m} n={n} k={k} pad={pad}", flush=True)
    full, ref, plan = _run(recipe, m, n, k, False, torch.float32, False, gpu, on=gpu, pad=pad)
    assert plan.startswith("mid ") and plan.endswith("split=1"), plan
    assert_linear_close(full, ref, f"{recipe} {m}x{n}x{k}")
    half, _, plan2 = _run(recipe, m, n, k, False, torch.bfloat16, False, gpu, on=gpu)
    assert plan == plan2 and torch.equal(half, full.to(torch.bfloat16))


@pytest.mark.parametrize("m,n,k", [(8, 130, 16), (100, 1000, 1040), (65, 257, 4096), (300, 2052, 2064)])
def test_medium_tiles_int8_exact(gpu, m, n, k):
    """The int32 sums are exact (4096 x 127^2 < 2^31): scales of one return them rounded to fp32."""
    from ayaka.kernel.hip import _lib, int8_scaled_mm

    g = torch.Generator().manual_seed(m + n + k)
    a = torch.randint(-127, 128, (m, k), generator=g, dtype=torch.int8)
    w = torch.randint(-127, 128, (n, k), generator=g, dtype=torch.int8)
    out = int8_scaled_mm(a.to(gpu), w.to(gpu).t(), torch.ones(m, device=gpu), torch.ones(n, device=gpu), out_dtype=torch.float32)
    assert _lib.last_plan().startswith("mid ")
    assert torch.equal(out.cpu(), (a.double() @ w.double().t()).float())


def test_medium_tiles_nan_codes_stay_in_their_row(gpu):
    """A NaN code (weight rows of 37 groups, so that the next row's codes follow a row's last
    stage at once) makes its own output column NaN and no other."""
    from ayaka.kernel.hip import mxfp8_scaled_mm

    m, n, k = 70, 140, 1184
    g = torch.Generator().manual_seed(5)
    a, w = _fp8((m, k), g).to(gpu), _fp8((n, k), g).to(gpu)
    ca = torch.full((m, k // 32), 120, dtype=torch.uint8, device=gpu)
    cb = torch.full((n, k // 32), 120, dtype=torch.uint8, device=gpu)
    cb[3, 0] = 0xFF
    y = mxfp8_scaled_mm(a, ca, w, cb, out=torch.empty(m, n, device=gpu))
    assert y[:, 3].isnan().all() and torch.isfinite(y[:, [c for c in range(n) if c != 3]]).all()


@pytest.mark.parametrize("stages", [1, 2, 3, 4, 5, 7, 8, 9])
@pytest.mark.parametrize("recipe", ["scaled", "block", "block16", "mx", "int8"])
def test_ring_stage_counts(gpu, recipe, stages):
    """Every remainder of the 64 x 64 ring's K loop, which runs in rounds of four 128-K stages, on
    shapes of one and of several tiles a side; 16-bit block scales start off a dword."""
    from ayaka.kernel.hip import _lib, fp8_blockwise_mm, int8_scaled_mm

    k = 128 * stages
    for m, n in ((70, 136), (200, 1028)):
        print(f"ring recipe={recipe} m={m} n={n} k={k}", flush=True)
        if recipe == "int8":
            g = torch.Generator().manual_seed(k + m)
            a, w = (torch.randint(-127, 128, (r, k), generator=g, dtype=torch.int8) for r in (m, n))
            out = int8_scaled_mm(a.to(gpu), w.to(gpu).t(), torch.ones(m, device=gpu), torch.ones(n, device=gpu), out_dtype=torch.float32)
            assert torch.equal(out.cpu(), (a.double() @ w.double().t()).float())
        elif recipe == "block16":
            g = torch.Generator().manual_seed(k + m)
            a, w = _fp8((m, k), g), _fp8((n, k), g)
            pool = (torch.rand(1 + m * stages, generator=g) * 1e-2 + 1e-3).to(torch.float16).to(gpu)
            poolb = (torch.rand(1 + -(-n // 128) * stages, generator=g) * 1e-2 + 1e-3).to(torch.bfloat16).to(gpu)
            sa, sb = pool[1:].view(m, stages), poolb[1:].view(-1, stages)
            out = fp8_blockwise_mm(a.to(gpu), w.to(gpu), sa, sb, out=torch.empty(m, n, dtype=torch.float32, device=gpu))
            ref = (a.to(gpu).double() * _expand(sa, m, k, 1, 128)) @ (w.to(gpu).double() * _expand(sb, n, k, 128, 128)).t()
            assert_linear_close(out, ref, f"block16 {m}x{n}x{k}")
        else:
            out, ref, _ = _run(recipe, m, n, k, True, torch.bfloat16, stages % 2 == 0, gpu)
            assert_linear_close(out, ref, f"{recipe} {m}x{n}x{k}")
        assert _lib.last_plan() == "mid 64x64 ring split=1", _lib.last_plan()


# One shape per tile, ragged on both sides, that keeps its tile up to K = 1536. N % 4 == 2 also
# keeps the 256 x 256 kernels away. Block scales have no 256 x 256 tile and one ring.
_TILES = {"256x256": (463, 28958), "128x128": (205, 28958), "128x64": (137, 16634), "128x128 ring": (205, 12358),
          "128x64 ring": (65, 8318), "64x64 ring": (65, 130)}
_TILE_SHAPES = {"scaled": _TILES, "int8": _TILES, "mx": _TILES | {"256x256": (403, 28390), "128x128": (205, 24718)}}
for _recipe in ("block", "block16"):
    _TILE_SHAPES[_recipe] = {"128x128": (205, 24718), "128x64": (65, 24718), "64x64 ring": (65, 130)}


@pytest.mark.parametrize("recipe,tile,m,n", [(r, t, *mn) for r, tiles in _TILE_SHAPES.items() for t, mn in tiles.items()])
def test_every_tile_and_stage_count(gpu, recipe, tile, m, n):
    """Each tile and ring with every remainder of its K loop (rounds of two or four stages), K
    tails and, for MXFP8, the three layouts of its codes: whole 512-K chunks (4, 8, 12 stages),
    whole dwords and unaligned."""
    less = {"scaled": (0, 48), "int8": (0, 112), "mx": (0, 32), "block": (0,), "block16": (0,)}[recipe]
    for stages in (*range(1, 10), 12):
        for k in (128 * stages - d for d in less):
            print(f"every tile recipe={recipe} tile={tile} m={m} n={n} k={k}", flush=True)
            out, ref, plan = _run(recipe, m, n, k, stages % 2 == 1, torch.bfloat16 if stages % 3 else torch.float32,
                                  stages % 2 == 0, gpu, on=gpu)
            assert plan == f"mid {tile} split=1", plan
            assert_linear_close(out, ref, f"{recipe} {m}x{n}x{k}")


@pytest.mark.parametrize("recipe,m,n,k,expect", [
    ("scaled", 205, 16634, 7792, "256x256 split=3"),
    ("scaled", 65, 16634, 7792, "128x128 split=3"),
    ("scaled", 137, 5486, 9872, "128x64 split=3"),
    ("scaled", 65, 8318, 5712, "128x128 ring split=3"),
    ("scaled", 65, 2690, 11952, "128x64 ring split=4"),
    ("scaled", 65, 130, 3632, "64x64 ring split=6"),
    ("block", 65, 16634, 3968, "128x128 split=3"),
    ("block", 65, 4158, 6656, "128x64 split=6"),
    ("block16", 65, 130, 2432, "64x64 ring split=4"),
    ("mx", 205, 16634, 6656, "256x256 split=3"),       # codes: whole chunks
    ("mx", 205, 16634, 7040, "256x256 split=3"),       # whole dwords
    ("mx", 205, 16634, 6336, "256x256 split=3"),       # unaligned
    ("mx", 65, 16634, 8192, "128x128 split=3"),
    ("mx", 65, 16634, 7808, "128x128 split=3"),
    ("mx", 65, 16634, 7232, "128x128 split=3"),
    ("mx", 137, 5486, 8192, "128x64 split=3"),
    ("mx", 137, 5486, 8576, "128x64 split=3"),
    ("mx", 137, 5486, 7904, "128x64 split=3"),
    ("mx", 65, 2690, 10240, "128x128 ring split=7"),
    ("mx", 65, 2690, 8960, "128x128 ring split=6"),
    ("mx", 65, 2690, 8800, "128x128 ring split=6"),
    ("mx", 65, 2690, 5632, "128x64 ring split=4"),
    ("mx", 65, 1346, 10880, "128x64 ring split=8"),
    ("mx", 65, 1346, 10816, "128x64 ring split=8"),
    ("mx", 65, 130, 2560, "64x64 ring split=3"),
    ("mx", 65, 130, 2816, "64x64 ring split=3"),
    ("mx", 65, 130, 2528, "64x64 ring split=3"),
])
def test_every_tile_split(gpu, recipe, m, n, k, expect):
    """K splits of each tile whose last piece is shorter."""
    print(f"tile split recipe={recipe} m={m} n={n} k={k}", flush=True)
    out, ref, plan = _run(recipe, m, n, k, True, torch.bfloat16, recipe == "block16", gpu, on=gpu)
    assert plan == f"mid {expect}", plan
    assert_linear_close(out, ref, f"{recipe} {m}x{n}x{k}")


_FAR = 1 << 23  # rows 8 MiB apart: 256 of them leave the medium tiles' 32-bit offsets


@pytest.mark.parametrize("recipe,m,n,k,bias,odt,far,expect", [
    ("scaled", 20, 300, 4224, True, torch.bfloat16, "a", "general 128x32 split=4"),   # last piece shorter
    ("scalar", 50, 260, 208, False, torch.float32, "a", "general 128x64 split=1"),    # K tail
    ("scaled", 130, 300, 4224, True, torch.float16, "a", "general 128x128 split=4"),
    ("scaled", 20, 140, 2176, False, torch.bfloat16, "w", "general 128x32 split=2"),
    ("block", 17, 300, 4096, True, torch.bfloat16, "a", "general 128x32 split=4"),    # bf16 weight scales
    ("block16", 40, 200, 4096, True, torch.float32, "a", "general 128x64 split=4"),   # fp16 activation scales too
    ("block", 129, 140, 1152, False, torch.bfloat16, "a", "general 128x128 split=1"),
    ("mx", 20, 300, 4224, True, torch.bfloat16, "a", "general 128x32 split=4"),
    ("mx", 64, 130, 1184, False, torch.float32, "a", "general 128x64 split=1"),       # unaligned codes
])
def test_general_kernel_rows_far_apart(gpu, recipe, m, n, k, bias, odt, far, expect):
    """Operand rows so far apart that the tiled kernels' offsets do not reach them."""
    print(f"general recipe={recipe} m={m} n={n} k={k} far={far}", flush=True)
    lda, ldw = (_FAR, None) if far == "a" else (None, _FAR)
    out, ref, plan = _run(recipe, m, n, k, bias, odt, recipe == "block" and m > 128, gpu, lda, ldw)
    assert plan == expect, plan
    assert_linear_close(out, ref, f"{recipe} {m}x{n}x{k}")


def test_general_kernel_int8_rows_far_apart(gpu):
    from ayaka.kernel.hip import _lib, int8_scaled_mm

    g = torch.Generator().manual_seed(3)
    for m, tile in ((20, 32), (50, 64), (130, 128)):
        a, w = (torch.randint(-127, 128, (r, 1040), generator=g, dtype=torch.int8) for r in (m, 260))
        out = int8_scaled_mm(_wide(a, _FAR, gpu), w.to(gpu).t(), torch.ones(m, device=gpu), torch.ones(260, device=gpu),
                             out_dtype=torch.float32)
        assert _lib.last_plan() == f"general 128x{tile} split=1", _lib.last_plan()
        assert torch.equal(out.cpu(), (a.double() @ w.double().t()).float())


@pytest.mark.parametrize("recipe,m,n,k,expect", [
    ("scaled", 32, 32900, 208, "general 128x32 split=1"),
    ("scaled", 33, 32900, 208, "mid 64x64 ring split=1"),
    ("scaled", 20, 32900, 640, "mid 64x64 ring split=1"),
    ("block", 17, 32900, 512, "general 128x32 split=1"),     # bf16 weight scales
    ("block", 1, 32900, 640, "general 128x32 split=1"),
    ("block16", 32, 32900, 896, "general 128x32 split=1"),
    ("block16", 32, 32900, 1024, "mid 64x64 ring split=1"),
    ("mx", 20, 32900, 640, "general 128x32 split=1"),
    ("block", 64, 32900, 384, "general 128x64 split=1"),
    ("block", 20, 16500, 128, "general 128x32 split=1"),
    ("block", 20, 16300, 128, "mid 64x64 ring split=1"),
    ("mx", 32, 17000, 224, "general 128x32 split=1"),
    ("mx", 32, 17000, 384, "mid 128x64 ring split=1"),
    ("mx", 20, 17000, 448, "general 128x32 split=1"),        # K % 128 != 0
    ("mx", 64, 32900, 128, "general 128x64 split=1"),
    ("mx", 8, 4100, 16512, "general 128x32 split=15"),
    ("mx", 9, 4900, 16512, "mid 128x64 ring split=6"),
    ("mx", 2, 18584, 4736, "general 128x32 split=3"),
    ("mx", 3, 1807, 12288, "skinny fn=1 fm=1 ks=4 g=2 ch=1 split=4"),
    ("mx", 2, 2048, 8192, "skinny fn=1 fm=1 ks=4 g=2 ch=4 split=4"),
    ("mx", 20, 4096, 10240, "mid 128x64 ring split=7"),
])
def test_decode_kernel_choice(gpu, recipe, m, n, k, expect):
    """Decode shapes at the edges between the general kernel's small tiles, the decode kernel
    and the medium tiles."""
    print(f"decode choice recipe={recipe} m={m} n={n} k={k}", flush=True)
    out, ref, plan = _run(recipe, m, n, k, True, torch.bfloat16, False, gpu)
    assert plan == expect, plan
    assert_linear_close(out, ref, f"{recipe} {m}x{n}x{k}")


@pytest.mark.parametrize("recipe,m,n,k,lda,expect", [
    ("scaled", 258, 3608, 10368, None, "pair split=8"),
    ("scaled", 258, 33136, 1536, None, "pair tail=3"),
    ("scaled", 64, 1302, 8192, None, "skinny"),
    ("scaled", 20, 300, 4224, _FAR, "general 128x32 split=4"),
    ("mx", 258, 3608, 7168, None, "pair split=7"),
    ("mx", 3, 1807, 12288, None, "skinny"),
    ("mx", 8, 4100, 16512, None, "general 128x32 split=15"),
    ("block", 258, 2184, 7296, None, "block256 split=7"),
    ("block", 258, 520, 16384, None, "block128 split=16"),
    ("block", 65, 1000, 4096, None, "mid 64x64 ring split=8"),
    ("block16", 40, 200, 4096, _FAR, "general 128x64 split=4"),
])
def test_launch_without_its_workspace(gpu, monkeypatch, recipe, m, n, k, lda, expect):
    """A launch that would split K and brings no workspace runs without the split."""
    from ayaka.kernel.hip import _lib

    print(f"no workspace recipe={recipe} m={m} n={n} k={k}", flush=True)
    _, _, plan = _run(recipe, m, n, k, False, torch.bfloat16, False, gpu, lda=lda)
    assert plan.startswith(expect) and "split=1" != plan.split()[-1], plan
    monkeypatch.setattr(_lib, "query", lambda name, *args: 0)
    out, ref, plan = _run(recipe, m, n, k, True, torch.bfloat16, False, gpu, lda=lda)
    assert plan.endswith("split=1"), plan
    assert_linear_close(out, ref, f"{recipe} {m}x{n}x{k}")


@pytest.mark.parametrize("recipe,m,n,k,expect", [
    ("scaled", 1794, 5888, 10752, "pair tail=1"),   # 115 us, its model just above the medium tiles'
    ("scaled", 1025, 3072, 1024, "mid 128x128 ring split=1"),
    ("block", 2328, 3456, 3328, "block256 split=1"),
    ("mx", 908, 8352, 2048, "pair tail=1"),
    ("mx", 700, 4096, 2048, "mid 128x128 ring split=1"),
])
def test_large_kernel_choice(gpu, recipe, m, n, k, expect):
    """Prefill shapes at the edge between the 256 x 256 kernels and the medium tiles."""
    print(f"large choice recipe={recipe} m={m} n={n} k={k}", flush=True)
    out, ref, plan = _run(recipe, m, n, k, True, torch.bfloat16, recipe == "block", gpu)
    assert plan == expect, plan
    assert_linear_close(out, ref, f"{recipe} {m}x{n}x{k}")


@pytest.mark.parametrize("recipe,m,n,k,odt,pad,expect", [
    ("scaled", 258, 33132, 1536, torch.bfloat16, 4, "pair tail=3"),    # padded output rows
    ("scaled", 258, 33132, 1536, torch.float32, 0, "pair tail=3"),
    ("scaled", 1300, 11712, 3072, torch.float16, 0, "pair tail=6"),    # a last round of 20 tiles
    ("scaled", 258, 8016, 128, torch.bfloat16, 0, "pair tail=1"),      # one pair of stages
    ("scaled", 520, 16388, 1280, torch.float16, 12, "pair tail=1"),
    ("scaled", 258, 3608, 10368, torch.bfloat16, 8, "pair split=8"),   # last piece shorter
    ("scaled", 258, 13252, 64, torch.float16, 4, "big"),               # one stage
    ("scaled", 516, 13260, 1088, torch.bfloat16, 4, "big"),
    ("int8", 258, 8016, 128, torch.float32, 4, "pair split=1"),
    ("int8", 520, 16388, 1280, torch.float32, 0, "pair split=1"),
    ("int8", 520, 16388, 1216, torch.float32, 4, "big"),
    ("mx", 258, 33132, 1536, torch.float16, 4, "pair tail=3"),
    ("mx", 1300, 11712, 3072, torch.bfloat16, 0, "pair tail=6"),
    ("mx", 258, 21904, 512, torch.float32, 4, "pair tail=1"),          # one chunk of codes
    ("mx", 520, 16388, 1024, torch.bfloat16, 12, "pair tail=1"),
    ("mx", 258, 3608, 7168, torch.bfloat16, 0, "pair split=7"),
    ("mx", 258, 1672, 20992, torch.float32, 0, "pair split=14"),       # last piece shorter
    ("block", 258, 1828, 128, torch.float32, 0, "block256 split=1"),   # one block
    ("block", 258, 1828, 8192, torch.float16, 4, "block256 split=8"),
    ("block", 258, 2184, 7296, torch.bfloat16, 0, "block256 split=7"),  # last piece shorter
    ("block", 258, 516, 16384, torch.bfloat16, 4, "block128 split=16"),
    ("block", 128, 26532, 3072, torch.float16, 4, "block128 split=1"),
])
@pytest.mark.parametrize("bias", [False, True])
def test_large_kernel_edges(gpu, recipe, m, n, k, odt, pad, expect, bias):
    """The 256 x 256 kernels' (and the block-scaled 128 x 128 one's) tails of M and N, first and
    last K steps, K splits, tail splits and strided outputs, on shapes that the dispatch gives
    them."""
    print(f"large edges recipe={recipe} m={m} n={n} k={k} out={odt} pad={pad} bias={bias}", flush=True)
    out, ref, plan = _run(recipe, m, n, k, bias, odt, recipe == "block" and bias, gpu, on=gpu, pad=pad)
    assert plan == expect, plan
    assert_linear_close(out, ref, f"{recipe} {m}x{n}x{k}")
    if recipe == "int8" and not bias:
        assert torch.equal(out, ref.float())
