"""The quantizers' GPU kernels against the torch operations the CPU path runs,
applied on the GPU: every byte and every scale the same, for each input type,
over magnitudes from denormal to the largest, all ties of the e2m1 grid, random
bit patterns, infinities and NaNs, and layouts that need a copy."""

import pytest
import torch

from gfx950_gluon_tutorials_amd import quant
from gfx950_gluon_tutorials_amd.gemm import _launch
from gfx950_gluon_tutorials_amd.gemm.prepared import PreparedGemm

pytestmark = pytest.mark.gpu


class _Plain(torch.Tensor):
    """A subclass keeps the torch operations."""


def _check(x):
    y = x.as_subclass(_Plain)
    for fn, bits in ((quant.quantize_mxfp4, torch.uint8), (quant.quantize_e5m2, torch.int32)):
        if fn is quant.quantize_mxfp4 and (x.dim() != 2 or x.shape[1] % 32):
            continue
        got, want = fn(x), [t.as_subclass(torch.Tensor) for t in fn(y)]
        assert got[0].dtype == want[0].dtype and got[1].shape == want[1].shape
        assert got[0].stride() == want[0].stride()
        assert torch.equal(got[0].view(torch.uint8), want[0].view(torch.uint8))
        assert torch.equal(got[1].view(bits), want[1].view(bits))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16, torch.float64])
@pytest.mark.parametrize("scale", [1.0, 1e-3, 3e4, 1e-38, 1e-42, 1e36])
def test_quantizers_random(gpu, dtype, scale):
    g = torch.Generator(device=gpu).manual_seed(1)
    for rows, K in ((1, 32), (333, 1056), (70, 8192)):
        _check((torch.randn(rows, K, generator=g, device=gpu, dtype=torch.float64) * scale).to(dtype))


@pytest.mark.parametrize("exponent", list(range(-140, 121, 13)) + [-126, -127, -11, 4, 9])
def test_quantizers_ties(gpu, exponent):
    g = torch.Generator(device=gpu).manual_seed(2)
    grid = torch.arange(256, device=gpu).double() / 32  # every e2m1 midpoint and its neighbours
    x = torch.cat([grid, -grid])[torch.randperm(512, generator=g, device=gpu)].reshape(4, 128)
    _check((x * 2.0 ** exponent).float())


def test_quantizers_bit_patterns(gpu):
    g = torch.Generator(device=gpu).manual_seed(3)
    b = torch.randint(-2**31, 2**31 - 1, (257, 1024), generator=g, device=gpu, dtype=torch.int64).int()
    for x in (b.view(torch.float32), b.view(torch.float16), b.view(torch.bfloat16)):
        _check(x)
        _check(torch.where(torch.isfinite(x), x, torch.zeros_like(x)))
    z = torch.zeros(3, 64, device=gpu)
    _check(z)
    for v in (float("inf"), -float("inf"), 1e-42, -0.0, float("nan")):
        z[1, 5] = v
        _check(z)


def test_quantizers_layouts(gpu):
    x = torch.randn(96, 256, device=gpu).bfloat16()
    _check(x.t())
    _check(x[:, 32:96])
    _check(x.reshape(-1)[1:1 + 64 * 255].reshape(255, 64))  # rows off the 16-byte grid
    _check(torch.randn(37, device=gpu))  # BF8 takes any shape
    _check(torch.randn(3, 5, 7, device=gpu).half())
    p, s = quant.quantize_mxfp4(torch.empty(0, 64, device=gpu))
    assert p.shape == (0, 32) and s.shape == (0, 2)
    with pytest.raises(RuntimeError):
        quant.quantize_e5m2(torch.empty(0, 64, device=gpu))  # no largest magnitude


def test_quantizers_leave_followed_tensors_to_torch(gpu):
    x = torch.randn(4, 64, device=gpu, requires_grad=True)
    assert quant.quantize_e5m2(x)[1].requires_grad
    with torch.no_grad():
        assert not quant.quantize_e5m2(x)[1].requires_grad
    w = torch.randn(3, 4, 64, device=gpu)
    p, s = torch.vmap(quant.quantize_mxfp4)(w)
    for i in range(3):
        a, b = quant.quantize_mxfp4(w[i])
        assert torch.equal(p[i], a) and torch.equal(s[i], b)
    with torch.autograd.forward_ad.dual_level():
        d = torch.autograd.forward_ad.make_dual(w[0], torch.ones_like(w[0]))
        assert torch.autograd.forward_ad.unpack_dual(quant.quantize_e5m2(d)[1]).tangent is not None


def test_e5m2_of_a_transposed_weight_is_read_in_place(gpu):
    """The codes of w.t() keep its strides, so they are the (K, N) operand of the
    BF8 GEMM as they are (a prepared launch refuses one that needs a copy)."""
    a, sa = quant.quantize_e5m2(torch.randn(48, 256, device=gpu))
    w = torch.randn(96, 256, device=gpu)
    b, sb = quant.quantize_e5m2(w.t())
    nk, sn = quant.quantize_e5m2(w)
    assert b.stride() == (1, 256) and torch.equal(b.t().view(torch.uint8), nk.view(torch.uint8)) and torch.equal(sb, sn)
    c, want = (torch.empty(48, 96, dtype=torch.bfloat16, device=gpu) for _ in range(2))
    PreparedGemm.a8w8([(a, b, c, sa, sb)])()
    _launch.gemm_a8w8(a, nk.t(), want, a_scale=sa, b_scale=sb)
    torch.cuda.synchronize()
    assert torch.equal(c, want)
