"""CPU check of the wrappers' direct launch path: it takes exactly the operands
the general path reads in place, over plain, padded, offset, sliced, transposed
and one-row layouts, and reads the same strides off them."""

import itertools

import pytest
import torch

from gfx950_gluon_tutorials_amd.gemm import _launch as L


def _views(rows, cols, dtype):
    """rows x cols views: contiguous, padded rows (aligned or not), a shifted base, transposed, every other column."""
    def raw(n):
        return torch.zeros(n, dtype=torch.uint8).view(dtype) if dtype is not torch.uint8 else torch.zeros(n, dtype=dtype)

    es = torch.empty(0, dtype=dtype).element_size()
    yield raw(rows * cols * es).reshape(rows, cols)
    for pad in (1, 4, 8, 16):
        yield raw(rows * (cols + pad) * es).reshape(rows, cols + pad)[:, :cols]
        yield raw((rows * cols + 16) * es)[pad // 2 : pad // 2 + rows * cols].reshape(rows, cols)
    yield raw(rows * cols * es).reshape(cols, rows).t()
    yield raw(rows * cols * 2 * es).reshape(rows, 2 * cols)[:, ::2]
    yield raw(cols * es).reshape(1, cols).expand(rows, cols)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float8_e5m2])
@pytest.mark.parametrize("M,N,K", [(1, 1, 16), (3, 5, 32), (16, 1, 24), (1, 40, 64)])
def test_direct_takes_what_the_general_path_reads_in_place(M, N, K, dtype):
    es = torch.empty(0, dtype=dtype).element_size()
    taken = 0
    for a, b in itertools.product(_views(M, K, dtype), _views(N, K, dtype)):
        c = torch.empty(M, N, dtype=torch.float16)
        d = L._direct(a, b.t(), c, es)
        assert (d is not None) == (L._rows_ok(a) and L._k_major_ok(b.t())), (a.stride(), b.stride())
        if d is not None:
            taken += 1
            assert d == (M, N, K, a.stride(0), b.stride(0), c.stride(), a.data_ptr(), b.data_ptr())
    assert taken
    assert L._direct(a, b.t(), torch.empty(M, N + 1, dtype=torch.float16), es) is None
    assert L._direct(a[None], b.t(), c, es) is None


@pytest.mark.parametrize("waves", [4, 8])
def test_direct_a4w4_scales(waves):
    M, N, K = 8, 12, 256
    a, b, c = (torch.zeros(M, K // 2, dtype=torch.uint8), torch.zeros(N, K // 2, dtype=torch.uint8), torch.empty(M, N))
    for sa, sb in itertools.product(_views(M, K // 32, torch.uint8), _views(N, K // 32, torch.uint8)):
        km = waves == 4 and L._kmajor_scales_ok(sa) and L._kmajor_scales_ok(sb)
        d = L._direct_a4w4(a, b, sa, sb, c, waves)
        assert (d is not None) == (km or (L._scales_ok(sa) and L._scales_ok(sb))), (sa.stride(), sb.stride())
        if d is not None:
            assert d[-4:] == (*sa.stride(), *sb.stride())
    assert L._direct_a4w4(a, b, sa[:-1], sb, c, waves) is None
    assert L._direct_a4w4(a, b[:, :-16], sa, sb, c, waves) is None
