"""The product's torch quantizers agree bit for bit with the oracle's numpy
restatement (CPU tensors)."""

import itertools

import numpy as np
import pytest
import torch

from gfx950_gluon_tutorials_amd import quant as Q
from oracle import gemm_ref as R


@pytest.mark.parametrize("seed,shape,scale", [(3, (64, 1024), 1.0), (5, (33, 256), 1e-3), (7, (8, 4096), 300.0)])
def test_mxfp4_matches_oracle(seed, shape, scale):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(shape, generator=g) * scale
    x[0, :32] = 0.0
    x[1, :32] = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0, 7.0] * 4)
    x[2, :32] = -x[1, :32]
    p, s = Q.quantize_mxfp4(x)
    po, so = R.quant_mxfp4(x.numpy())
    np.testing.assert_array_equal(p.numpy(), po)
    np.testing.assert_array_equal(s.numpy(), so)
    np.testing.assert_array_equal(Q.dequantize_mxfp4(p, s).numpy(), R.mxfp4_dequant(po, so))


@pytest.mark.parametrize("seed,scale", [(2, 1.0), (9, 1e-4), (11, 1e3)])
def test_e5m2_matches_oracle(seed, scale):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(128, 512, generator=g) * scale
    q, s = Q.quantize_e5m2(x)
    qo, so = R.quant_e5m2_per_tensor(x.numpy())
    np.testing.assert_array_equal(q.view(torch.uint8).numpy(), qo)
    assert float(s) == float(so)


def test_mxfp4_rejects_ragged_k():
    with pytest.raises(ValueError):
        Q.quantize_mxfp4(torch.zeros(4, 40))


def test_kernel_input_resolves_negation():
    """The GPU kernels read memory, where a lazily negated view holds the opposite values."""
    x = torch.randn(2, 32, generator=torch.Generator().manual_seed(0))
    y = Q._kernel_input(torch._neg_view(x))
    assert not y.is_neg() and torch.equal(y, -x)


def _layouts():
    """3-D and 2-D views: every order of dimensions, dense, sliced, stepped, broadcast, shifted off the 16-byte grid."""
    g = torch.Generator().manual_seed(1)
    r = lambda *shape: torch.randn(*shape, generator=g)
    for p in itertools.permutations(range(3)):
        yield r(3, 4, 8).permute(p)
        yield r(3, 1, 8).permute(p)
        yield r(3, 4, 16)[:, :, :8].permute(p)
        yield r(3, 4, 16)[:, :, ::2].permute(p)
        yield r(3, 1, 8).expand(3, 4, 8).permute(p)
    yield r(6, 8).t()
    yield r(6, 8)[:, 2:3]
    yield r(1 + 48)[1:].reshape(6, 8).t()
    yield r(2, 3, 4, 5).contiguous(memory_format=torch.channels_last)
    yield torch._neg_view(r(6, 8).t())
    yield r(1)[0]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16, torch.float64])
def test_e5m2_buffers_keep_the_layout_of_the_torch_operations(dtype):
    for x in _layouts():
        x = torch._neg_view(torch._neg_view(x).to(dtype)) if x.is_neg() else x.to(dtype)
        src, codes = Q._e5m2_buffers(x)
        want, _ = Q.quantize_e5m2(x)  # on the CPU: the torch operations
        assert codes.shape == want.shape and codes.stride() == want.stride(), (x.shape, x.stride())
        assert src.stride() == codes.stride() and src.dtype in Q._IN and src.data_ptr() % 16 == 0
        assert not src.is_neg() and torch.equal(src, x.to(src.dtype))
