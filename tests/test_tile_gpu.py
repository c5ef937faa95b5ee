"""The small output tiles of the data-parallel schedule (16x16 to 256x128, for
grids that 256x256 tiles would leave the chip idle on) against stream-K, whose
256x256 tiles accumulate every element by the same MFMA sequence: bit for bit.

One shape per tile and operand size, named by the tile the launch picks there
(256 CUs): just past the tile's edges in M and N, a K tail where the type
allows one, and more stages than the tile's LDS ring has slots.  C is a column
slice of a wider buffer, whose padding must survive.
"""

import pytest
import torch

import launched
import tile_pick
from gfx950_gluon_tutorials_amd import quant
from gfx950_gluon_tutorials_amd.gemm import _launch

pytestmark = pytest.mark.gpu

SHAPES16 = {"16x16": (4, 1, 2024), "16x32": (2055, 17, 992), "32x32": (2106, 37, 776), "64x32": (2055, 34, 472),
            "64x64": (193, 2065, 400), "128x64": (514, 1798, 648), "128x128": (1089, 1815, 456),
            "256x128": (2256, 2285, 264)}
SHAPES8 = {"16x16": (1, 14, 2832), "16x32": (17, 2291, 1856), "32x32": (2101, 37, 1440), "64x32": (1634, 131, 912),
           "64x64": (208, 2117, 784), "128x64": (449, 2076, 1312), "128x128": (1685, 1168, 784),
           "256x128": (1805, 2248, 528)}
SHAPES4 = {"16x16": (3, 9, 4864), "16x32": (2051, 17, 3584), "32x32": (2136, 35, 2560), "64x32": (2082, 101, 2048),
           "64x64": (195, 2125, 1536), "128x64": (517, 1796, 1536), "128x128": (1671, 1164, 1536),
           "256x128": (1798, 2246, 1280)}
TILES = list(SHAPES16)


def _out(gpu, M, N, dtype):
    buf = torch.full((M, N + 3), float("nan"), dtype=dtype, device=gpu)
    return buf, buf[:, :N]


def _same(buf, c, want):
    torch.cuda.synchronize()
    assert torch.equal(c.contiguous().view(torch.int16), want.view(torch.int16))
    assert torch.isnan(buf[:, c.shape[1]:]).all()


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tile", TILES)
def test_a16w16_tile_bits(gpu, tile, dtype, waves):
    M, N, K = SHAPES16[tile]
    print(f"\n[case] a16w16 {tile} {M}x{N}x{K} {dtype} {waves}w", flush=True)
    g = torch.Generator(device=gpu).manual_seed(M + N)
    a = torch.randn(M, K, generator=g, device=gpu).to(dtype)
    b = torch.randn(N, K, generator=g, device=gpu).to(dtype)
    buf, c = _out(gpu, M, N, dtype)
    launched.a16w16(tile, a, b.T, c, waves=waves)
    _launch.gemm_a16w16(a, b.T, c, waves=waves)
    want = _launch.gemm_a16w16(a, b.T, torch.empty(M, N, dtype=dtype, device=gpu), schedule="streamk", waves=waves)
    _same(buf, c, want)


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("out", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tile", TILES)
def test_a8w8_tile_bits(gpu, tile, out, waves):
    M, N, K = SHAPES8[tile]
    print(f"\n[case] a8w8 {tile} {M}x{N}x{K} {out} {waves}w", flush=True)
    g = torch.Generator(device=gpu).manual_seed(M + N)
    a, sa = quant.quantize_e5m2(torch.randn(M, K, generator=g, device=gpu))
    b, sb = quant.quantize_e5m2(torch.randn(N, K, generator=g, device=gpu))
    buf, c = _out(gpu, M, N, out)
    launched.a8w8(tile, a, b.T, c, waves=waves)
    _launch.gemm_a8w8(a, b.T, c, a_scale=sa, b_scale=sb, waves=waves)
    want = _launch.gemm_a8w8(a, b.T, torch.empty(M, N, dtype=out, device=gpu), a_scale=sa, b_scale=sb,
                             schedule="streamk", waves=waves)
    _same(buf, c, want)


def _k_major(s):
    buf = torch.full((s.shape[1], -(-s.shape[0] // 4) * 4), 127, dtype=torch.uint8, device=s.device)
    buf[:, :s.shape[0]] = s.t()
    return buf.t()[:s.shape[0]]


@pytest.mark.parametrize("layout", ["row", "kmajor", "preshuffled"])
@pytest.mark.parametrize("tile", TILES)
def test_a4w4_tile_bits(gpu, tile, layout):
    M, N, K = SHAPES4[tile]
    if layout == "kmajor":  # the last group's rows end inside a dword, for A and for B
        M, N = M | 1, N | 3
    print(f"\n[case] a4w4 {tile} {M}x{N}x{K} {layout}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(M + N)
    a, sa = quant.quantize_mxfp4(torch.randn(M, K, generator=g, device=gpu))
    b, sb = quant.quantize_mxfp4(torch.randn(N, K, generator=g, device=gpu))
    want = _launch.gemm_a4w4(a, b, sa, sb, torch.empty(M, N, dtype=torch.bfloat16, device=gpu), schedule="streamk")
    if layout == "kmajor":
        sa, sb = _k_major(sa), _k_major(sb)
    elif layout == "preshuffled":
        sa, sb = quant.preshuffle_e8m0(sa), quant.preshuffle_e8m0(sb)
    buf, c = _out(gpu, M, N, torch.bfloat16)
    launched.a4w4(tile, a, b, sa, sb, c)
    _launch.gemm_a4w4(a, b, sa, sb, c)
    _same(buf, c, want)


def _spread(x, stride):
    """x's rows `stride` bytes apart."""
    es = x.element_size()
    buf = torch.empty(x.shape[0] * stride // es, dtype=x.dtype, device=x.device)
    wide = buf.as_strided(x.shape, (stride // es, 1))
    wide.copy_(x)
    return wide


# Row strides from where 256 rows stop fitting a 2^31-byte buffer range (the
# 256x128 tile, which these shapes take with packed rows) to the largest the
# library takes; K tails need a stride below that.
@pytest.mark.parametrize("stride", [2**23 - 16, 2**23, 2**24 - 16, 2**24])
@pytest.mark.parametrize("op", ["f16", "bf8", "mxfp4", "mxfp4_scales"])
def test_wide_rows(gpu, op, stride):
    M, N = 1537, 4096
    K = {"f16": 1024 - 8, "bf8": 1024 - 16}.get(op, 1024)
    if stride == 2**24 and not op.startswith("mxfp4"):
        K = 1024
    print(f"\n[case] wide rows {op} {M}x{N}x{K} stride {stride}", flush=True)
    kind = op.split("_")[0]
    assert tile_pick.dense(kind, M, N, K) == "256x128"
    if op != "mxfp4_scales":
        assert (tile_pick.dense(kind, M, N, K, lda=stride) == "256x128") == (stride < 2**23)
    g = torch.Generator(device=gpu).manual_seed(K)
    a = torch.randn(M, K, generator=g, device=gpu)
    b = torch.randn(N, K, generator=g, device=gpu)
    out = [torch.empty(M, N, dtype=torch.float16, device=gpu) for _ in range(2)]
    if op == "f16":
        a, b = a.half(), b.half()
        for c, x in zip(out, (a, _spread(a, stride))):
            _launch.gemm_a16w16(x, b.T, c)
    elif op == "bf8":
        a, b = a.to(torch.float8_e5m2), b.to(torch.float8_e5m2)
        for c, x in zip(out, (a, _spread(a, stride))):
            _launch.gemm_a8w8(x, b.T, c)
    else:
        (a, sa), (b, sb) = quant.quantize_mxfp4(a), quant.quantize_mxfp4(b)
        wide = (a, _spread(sa, stride)) if op == "mxfp4_scales" else (_spread(a, stride), sa)
        for c, (x, s) in zip(out, ((a, sa), wide)):
            _launch.gemm_a4w4(x, b, s, sb, c)
    torch.cuda.synchronize()
    assert torch.equal(out[0].view(torch.int16), out[1].view(torch.int16))
