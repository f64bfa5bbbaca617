"""GPU: the tiled W8A16 GEMM at the edges of its tiles, K stages and K splits, against the
fp64 product of the same operands, and the launch rule's choice for each.

Bound per element, with u the unit roundoff of the activation type (2^-p for p significand
bits: 2^-8 for bf16, 2^-11 for fp16) and S = sum |x w s|:

* each w s is rounded to the activation type, u S (in fp16 also half a subnormal step,
  2^-25 sum |x|);
* the fp32 sum, at most (K + 2) 2^-24 S, and the output's rounding, u |y|.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu
FP8 = torch.float8_e4m3fn
UNIT = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}


def _operands(m, n, k, xdt, by, bx, sdt, dev):
    g = torch.Generator().manual_seed(m * 31 + n * 7 + k)
    w = (torch.randn(n, k, generator=g) * 60).clamp(-448, 448).to(FP8)
    x = torch.randn(m, k, generator=g).to(xdt)
    shape = (-(-n // by), -(-k // bx))
    if sdt == "e8m0":
        scale = torch.randint(110, 124, shape, generator=g, dtype=torch.uint8)
        value = torch.exp2(scale.double() - 127)
    else:
        scale = (torch.rand(shape, generator=g) * 3e-4 + 1e-5).to(getattr(torch, sdt))
        value = scale.double()
    full = value.repeat_interleave(by, 0)[:n].repeat_interleave(bx, 1)[:, :k]
    return x.to(dev), w.to(dev), scale.to(dev), full.to(dev)


def _check(m, n, k, xdt, by, bx, sdt, dev):
    """One call within the bound; returns its recorded plan."""
    from ayaka.kernel.hip import _lib, fp8_weight_only_gemm

    bx = k if bx is None else bx
    print(f"w8a16 m={m} n={n} k={k} x={xdt} by={by} bx={bx} scale={sdt}", flush=True)
    x, w, scale, full = _operands(m, n, k, xdt, by, bx, sdt, dev)
    y = fp8_weight_only_gemm(x, w, scale, scale.shape[1], by, bx, sdt).double()
    plan = _lib.last_plan()
    ws = w.double() * full
    ref, mag = x.double() @ ws.t(), x.double().abs() @ ws.abs().t()
    u = UNIT[xdt]
    bound = u * ref.abs() + (u + (k + 2) * 2.0**-24) * mag
    if xdt == torch.float16:
        bound = bound + 2.0**-25 * x.double().abs().sum(1, keepdim=True)
    worst = ((y - ref).abs() / bound.clamp_min(1e-30)).max().item()
    assert worst <= 1.01, worst  # 1% for second-order terms
    return plan


@pytest.mark.parametrize("m,n,k,xdt,by,bx,sdt,plan", [
    (33, 129, 16, torch.bfloat16, 1, None, "float32", "128x64 split=1"),      # one short stage
    (64, 128, 64, torch.float16, 1, None, "float32", "128x64 split=1"),       # exact tile and stage
    (65, 257, 1040, torch.bfloat16, 1, None, "bfloat16", "128x64 split=1"),   # every remainder
    (20, 1000, 1936, torch.float16, 1, None, "float32", "128x64 split=3"),    # K no decode kernel takes, last piece shorter
    (40, 2051, 3072, torch.bfloat16, 1, None, "float32", "128x64 split=6"),   # N not a multiple of 4, split
    (1, 300, 144, torch.bfloat16, 1, None, "e8m0", "128x64 split=1"),
    (200, 4099, 14336, torch.float16, 1, None, "float32", "256x256 split=12"),
    (129, 9000, 7168, torch.bfloat16, 128, 128, "float32", "256x256 split=6"),
    (500, 5000, 4096, torch.bfloat16, 1, None, "float32", "128x128 split=3"),
    (257, 513, 336, torch.bfloat16, 64, 128, "float32", "128x64 split=1"),
    (300, 640, 4160, torch.float16, 128, 64, "bfloat16", "128x64 split=8"),
    (1000, 28672, 1040, torch.bfloat16, 1, None, "float32", "256x256 split=1"),
    (2049, 8200, 576, torch.float16, 1, None, "float32", "128x128 split=1"),
    (65, 16634, 8320, torch.bfloat16, 1, None, "float32", "256x128 split=6"),
    (65, 16634, 8320, torch.float16, 128, 128, "float32", "256x128 split=6"),
    (65, 4158, 8320, torch.float16, 128, 192, "float32", "128x128 split=12"),  # scale blocks of three stages
])
def test_weight_only_gemm_tile(gpu, m, n, k, xdt, by, bx, sdt, plan):
    got = _check(m, n, k, xdt, by, bx, sdt, gpu)
    assert got == f"w8a16 tile {plan}", got


@pytest.mark.parametrize("tile,m,n", [("256x256", 403, 24718), ("256x128", 529, 21946), ("128x128", 205, 24718),
                                      ("128x64", 65, 130)])
@pytest.mark.parametrize("by,bx", [(1, None), (128, 64), (96, 128)])
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16])
def test_weight_only_gemm_every_tile(gpu, tile, m, n, by, bx, xdt):
    """One to five K stages and tails on each tile, ragged on both sides."""
    for k in (16, 64, 112, 128, 192, 208, 320):
        got = _check(m, n, k, xdt, by, bx, "float32", gpu)
        assert got == f"w8a16 tile {tile} split=1", got


@pytest.mark.parametrize("m,n,k,bx,plan", [
    (32, 3840, 3200, None, "w8a16 tile 128x64 split=6"),
    (25, 3840, 3200, None, "w8a16 tile 128x64 split=6"),
    (24, 3840, 3200, None, "w8a16 skinny split=13"),
    (31, 640, 14464, None, "w8a16 skinny split=57"),  # few 128-row tiles
    (32, 3840, 3200, 128, "w8a16 skinny split=13"),   # block scales
])
def test_weight_only_gemm_decode_choice(gpu, m, n, k, bx, plan):
    """Batches of 17 to 32 rows whose K only the skinny kernel or the tiled one takes (an odd
    multiple of 128), at the edges of the rule between the two."""
    got = _check(m, n, k, torch.bfloat16, 1 if bx is None else 128, bx, "float32", gpu)
    assert got == plan, got


@pytest.mark.parametrize("m,n,k", [(24, 3840, 3200), (16, 512, 8192), (30, 1280, 17664), (40, 2051, 3072), (200, 4099, 14336)])
def test_weight_only_gemm_without_its_workspace(gpu, monkeypatch, m, n, k):
    """A launch that would split K and brings no workspace runs without the split."""
    from ayaka.kernel.hip import _lib

    assert not _check(m, n, k, torch.bfloat16, 1, None, "float32", gpu).endswith("split=1")
    monkeypatch.setattr(_lib, "query", lambda name, *args: 0)
    plan = _check(m, n, k, torch.bfloat16, 1, None, "float32", gpu)
    assert plan.startswith("w8a16 tile") and plan.endswith("split=1"), plan


def test_weight_only_gemm_tile_all_codes_and_special_scales(gpu):
    """Every weight code against a one-hot activation: the weight times its row's scale,
    rounded to bf16, NaN codes included; tiny and huge scales."""
    from ayaka.kernel.hip import fp8_weight_only_gemm

    codes = torch.arange(256, dtype=torch.uint8, device=gpu)
    scales = torch.tensor([1.0, 0.3, 2.0**-100, 1e-30, 1.7e30, 3.0], device=gpu)
    w = codes.repeat(scales.numel(), 1)  # row r: every code, scale r
    x = torch.eye(256, device=gpu, dtype=torch.bfloat16)
    y = fp8_weight_only_gemm(x, w, scales.reshape(-1, 1), 1, 1, 256, "float32")
    values = codes.view(FP8).float()
    ref = values[:, None] * scales
    nan_rows = values.isnan().nonzero().flatten()
    # a NaN weight meets a zero activation in every other row: all outputs of its column are NaN
    assert nan_rows.numel() == 2 and y.isnan().all()
    w[:, nan_rows] = 0
    ref[nan_rows] = 0.0
    y = fp8_weight_only_gemm(x, w, scales.reshape(-1, 1), 1, 1, 256, "float32")
    assert torch.equal(y, ref.to(torch.bfloat16))


def test_weight_only_gemm_tile_views_and_graph(gpu):
    """Strided activation, output view with an odd stride, and a captured K-split launch."""
    from ayaka.kernel.hip import fp8_weight_only_gemm

    m, n, k = 70, 514, 2048
    x, w, scale, full = _operands(m, n, k, torch.bfloat16, 1, k, "float32", gpu)
    wide = torch.zeros(m, k + 24, dtype=x.dtype, device=gpu)
    wide[:, :k] = x
    wide[:, k:] = torch.nan
    ref = fp8_weight_only_gemm(x, w, scale, 1, 1, k, "float32")
    out = torch.full((m, n + 3), 7.0, dtype=x.dtype, device=gpu)
    fp8_weight_only_gemm(wide[:, :k], w, scale, 1, 1, k, "float32", out=out[:, :n])
    assert torch.equal(out[:, :n], ref) and (out[:, n:] == 7).all()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = fp8_weight_only_gemm(x, w, scale, 1, 1, k, "float32")
    for i in range(3):
        captured.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, ref), i
        torch.mm(torch.ones(64, 64, device=gpu), torch.ones(64, 64, device=gpu))


def test_weight_only_gemm_empty_k_is_refused(gpu):
    """An empty K is an argument error, also for callers that give the scale layout."""
    from ayaka.kernel.hip import fp8_weight_only_gemm

    x, w = torch.empty(2, 0, dtype=torch.bfloat16, device=gpu), torch.empty(128, 0, device=gpu).to(FP8)
    with pytest.raises(ValueError, match="bad shape"):
        fp8_weight_only_gemm(x, w, torch.ones(128, device=gpu), 1, 1, 128, "float32")
