"""Grouped GEMMs on every output tile, 16x16 to 256x256: each expert's rows equal,
bit for bit, stream-K's on that expert's slice (256x256 tiles, the same MFMA
sequence); rows past the last expert's stay as they were.  Each shape names the
tile that the launch picks there (256 CUs), and has experts of more than one
tile's rows and a last column tile that is not full.

E past 64 takes the expert lookup through more than one pass; empty experts,
one-row experts and experts just past a tile's rows are in every table."""

import numpy as np
import pytest
import torch

import tile_pick
from gfx950_gluon_tutorials_amd import quant
from gfx950_gluon_tutorials_amd.gemm import _launch
from gfx950_gluon_tutorials_amd.gemm.moe import moe_matmul, moe_matmul_a4w4, moe_matmul_a8w8

pytestmark = pytest.mark.gpu


def _counts(E, mean, seed):
    rng = np.random.default_rng(seed)
    c = rng.multinomial(mean * E, rng.dirichlet([2.0] * E))
    c[0], c[E // 2], c[-1] = 0, 1, mean + 1
    return c


# (E, mean rows, N, K, tile)
ALL = [(70, 3, 136, 512, "64x64"), (9, 17, 1032, 2048, "64x64"), (130, 40, 264, 768, "64x64"),
       (6, 150, 520, 1024, "64x64")]
SHAPES16 = [(3, 16, 24, 512, "16x16"), (4, 86, 360, 512, "16x32"), (6, 79, 304, 576, "32x32"), (4, 33, 56, 320, "64x32"),
            (5, 154, 824, 256, "64x64"), (4, 378, 984, 768, "128x64"), (5, 209, 3144, 256, "128x128"),
            (66, 230, 520, 512, "128x128"), (6, 909, 1296, 256, "256x128"), (12, 462, 1656, 256, "256x256"),
            (66, 230, 1032, 256, "256x256")]
SHAPES8 = [(4, 8, 56, 512, "16x16"), (4, 86, 296, 1152, "16x32"), (4, 49, 432, 512, "32x32"), (5, 115, 592, 512, "64x32"),
           (4, 169, 1008, 512, "64x64"), (6, 361, 520, 1408, "128x64"), (5, 389, 2200, 512, "128x128"),
           (9, 534, 1264, 512, "256x128"), (6, 1017, 1720, 512, "256x256")]
SHAPES4 = [(4, 22, 24, 1024, "16x16"), (4, 111, 248, 2048, "16x32"), (3, 78, 664, 1024, "32x32"),
           (6, 61, 680, 1024, "64x32"), (5, 168, 688, 1280, "64x64"), (4, 426, 792, 1792, "128x64"),
           (4, 819, 792, 1280, "128x128"), (6, 470, 2280, 1024, "256x128"), (9, 284, 2968, 1024, "256x256")]
CASES = [(kind, *s) for kind, shapes in (("f16", SHAPES16), ("bf16", SHAPES16), ("bf8", SHAPES8), ("mxfp4", SHAPES4))
         for s in ALL + shapes]


@pytest.mark.parametrize("kind,E,mean,N,K,tile", CASES)
def test_moe_tile_bits(gpu, kind, E, mean, N, K, tile):
    counts = _counts(E, mean, E + N)
    off = np.concatenate([[0], np.cumsum(counts)])
    T = int(off[-1]) + 5  # rows no expert owns
    print(f"\n[case] moe {kind} E={E} T={T} N={N} K={K} {tile}", flush=True)
    assert tile_pick.moe(kind, T, E, N, K) == tile
    g = torch.Generator(device=gpu).manual_seed(E)
    offs = torch.tensor(off, dtype=torch.int32, device=gpu)
    x = torch.randn(T, K, generator=g, device=gpu)
    w = torch.randn(E, N, K, generator=g, device=gpu)
    dt = torch.float16 if kind == "f16" else torch.bfloat16
    c = torch.full((T, N), 7.0, dtype=dt, device=gpu)
    if kind in ("f16", "bf16"):
        a, b = x.to(dt), w.to(dt)
        moe_matmul(a, b, offs, c)
        one = lambda r, e, o: _launch.gemm_a16w16(a[r], b[e].T, o, schedule="streamk")
    elif kind == "bf8":
        a, sa = quant.quantize_e5m2(x)
        qs = [quant.quantize_e5m2(w[e]) for e in range(E)]
        b, sb = torch.stack([q for q, _ in qs]), torch.cat([s for _, s in qs])
        moe_matmul_a8w8(a, b, offs, c, a_scale=sa, b_scales=sb)
        one = lambda r, e, o: _launch.gemm_a8w8(a[r], b[e].T, o, a_scale=sa, b_scale=sb[e:e + 1], schedule="streamk")
    else:
        a, sa = quant.quantize_mxfp4(x)
        b, sb = (t.reshape(E, N, -1) for t in quant.quantize_mxfp4(w.reshape(E * N, K)))
        moe_matmul_a4w4(a, b, sa, sb, offs, c)
        one = lambda r, e, o: _launch.gemm_a4w4(a[r], b[e], sa[r], sb[e], o, schedule="streamk")
    for e in range(E):
        if counts[e]:
            r = slice(int(off[e]), int(off[e + 1]))
            want = one(r, e, torch.empty(int(counts[e]), N, dtype=dt, device=gpu))
            assert torch.equal(c[r].view(torch.int16), want.view(torch.int16)), f"expert {e}"
    torch.cuda.synchronize()
    assert torch.all(c[int(off[-1]):] == 7.0)


@pytest.mark.parametrize("E", [64, 65, 512, 577, 4097, 5000])
def test_many_experts(gpu, E):
    """One expert per lane of the lookup, several, more than its batch of loads and more than
    64 (a second pass of more than one chunk), with empty experts: small integers, whose
    products are exact, against torch in fp32."""
    T, N, K = 2 * E + 3, 24, 64
    print(f"\n[case] moe f16 E={E} T={T} N={N} K={K}", flush=True)
    rng = np.random.default_rng(E)
    counts = rng.multinomial(2 * E, rng.dirichlet([0.5] * E))
    owner = torch.from_numpy(np.repeat(np.arange(E), counts)).to(gpu)
    offs = torch.from_numpy(np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)).to(gpu)
    g = torch.Generator(device=gpu).manual_seed(E)
    a = torch.randint(-2, 3, (T, K), generator=g, device=gpu).half()
    b = torch.randint(-2, 3, (E, N, K), generator=g, device=gpu).half()
    c = torch.full((T, N), 7.0, dtype=torch.float16, device=gpu)
    moe_matmul(a, b, offs, c)
    want = (a[:2 * E, None].float() * b[owner].float()).sum(-1)
    torch.cuda.synchronize()
    assert torch.equal(c[:2 * E].float(), want)
    assert torch.all(c[2 * E:] == 7.0)
