"""CPU checks of the grouped (MoE) GEMM: argument validation of the C ABI
(status codes returned before any launch), kernel names, and a restatement
of the kernel's expert lookup (g9_gemm.hpp moe_find, with the grid of
g9_capi.hip launch_moe) at every tile height, with up to and past one expert
per lane, showing that any offset table keeps every access inside A, C and the
experts' B, and that valid tables give each expert's rows to exactly one tile."""

import re

import numpy as np
import pytest

from gfx950_gluon_tutorials_amd import _lib
from gfx950_gluon_tutorials_amd.gemm.moe import KERNEL_NAME

FAKE = 0x10000


def _moe16(T=512, N=256, K=256, E=4, sam=None, sbn=None, sbe=None, scm=None, dtype=_lib.G9_F16, off=FAKE):
    lib = _lib.load()
    return lib.g9_moe_a16w16(FAKE, FAKE, FAKE, off, T, N, K, E, K if sam is None else sam,
                             K if sbn is None else sbn, N * K * 2 if sbe is None else sbe,
                             N if scm is None else scm, dtype, None)


@pytest.mark.parametrize("kw,code", [
    (dict(E=0), _lib.G9_ERR_SHAPE),
    (dict(T=-1), _lib.G9_ERR_SHAPE),
    (dict(K=100), _lib.G9_ERR_SHAPE),
    (dict(N=0), _lib.G9_ERR_SHAPE),
    (dict(off=0), _lib.G9_ERR_LAYOUT),
    (dict(off=FAKE + 2), _lib.G9_ERR_LAYOUT),
    (dict(sbe=8), _lib.G9_ERR_LAYOUT),
    (dict(sam=100), _lib.G9_ERR_LAYOUT),
    (dict(scm=100), _lib.G9_ERR_LAYOUT),
    (dict(dtype=_lib.G9_FP4), _lib.G9_ERR_DTYPE),
    (dict(T=0), _lib.G9_OK),  # no tokens: nothing to launch
    (dict(T=0, K=100), _lib.G9_ERR_SHAPE),
])
def test_moe_a16w16_argument_validation(kw, code):
    assert _moe16(**kw) == code


def test_moe_a4w4_argument_validation():
    lib = _lib.load()
    T, N, K, E = 512, 256, 512, 4

    def call(out=_lib.G9_BF16, sasm=K // 32, sbse=N * K // 32, asc=FAKE):
        return lib.g9_moe_a4w4(FAKE, FAKE, FAKE, asc, FAKE, FAKE, T, N, K, E, K // 2, K // 2, N * K // 2,
                               sasm, K // 32, sbse, N, out, None)

    assert call(out=_lib.G9_BF8) == _lib.G9_ERR_DTYPE
    assert call(sasm=K // 32 - 4) == _lib.G9_ERR_LAYOUT
    assert call(sbse=6) == _lib.G9_ERR_LAYOUT
    assert call(asc=0) == _lib.G9_ERR_LAYOUT


def test_moe_a8w8_argument_validation():
    lib = _lib.load()
    T, N, K, E = 512, 256, 512, 4

    def call(out=_lib.G9_BF16, K_=K, sb=FAKE):
        return lib.g9_moe_a8w8(FAKE, FAKE, FAKE, FAKE, None, sb, T, N, K_, E, K_, K_, N * K_, N, out, None)

    assert call(out=_lib.G9_FP4) == _lib.G9_ERR_DTYPE
    assert call(K_=192) == _lib.G9_ERR_SHAPE  # K must be a multiple of 128
    assert call(sb=FAKE + 2) == _lib.G9_ERR_LAYOUT


def test_moe_kernel_names():
    pairs = [(_lib.G9_F16, _lib.G9_F16), (_lib.G9_BF16, _lib.G9_BF16), (_lib.G9_BF8, _lib.G9_BF16),
             (_lib.G9_BF8, _lib.G9_F16), (_lib.G9_FP4, _lib.G9_BF16), (_lib.G9_FP4, _lib.G9_F16)]
    names = {_lib.moe_kernel_name(dt, out) for dt, out in pairs}
    assert len(names) == 6 and all(n and n.endswith("_moe_4w") for n in names)
    # The profiler filter takes the grouped kernels of every tile, and only those.
    with open(_lib.LIB_PATH, "rb") as fh:
        built = {n.decode() for n in re.findall(rb"\bg9_[a-z0-9_]+(?:_[48]w|_t\d+x\d+)\b", fh.read())}
    grouped = {n for n in built if KERNEL_NAME in n}
    assert names | {f"g9_{op}_moe_t{tm}x{tn}" for op in ("a16w16_f16", "a16w16_bf16", "a8w8", "a4w4")
                    for tm, tn in ((16, 16), (16, 32), (32, 32), (64, 32), (64, 64), (128, 64), (128, 128), (256, 128))} \
        == grouped
    assert not any("_dp_" in n or "_sk" in n or "_splitk_" in n for n in grouped)
    assert _lib.moe_kernel_name(_lib.G9_F16, _lib.G9_BF16) is None


TILES = [16, 32, 64, 128, 256]
XCDS, GROUP_M = 8, 4


def grid_m(T, E, tile):
    """The launch's m-tiles (g9_capi.hip launch_moe): at most min(E, T) experts have rows."""
    return (T + min(E, T) * (tile - 1)) // tile


def tile_coords(pid, grid, tiles_m, tiles_n):
    """Restatement of g9_common.hpp tile_coords: contiguous ranges to XCDs, then groups of GROUP_M m-tiles."""
    per, tall = -(-grid // XCDS), grid % XCDS or XCDS
    xcd, local = pid % XCDS, pid // XCDS
    pid = xcd * per + local if xcd < tall else tall * per + (xcd - tall) * (per - 1) + local
    first = pid // (GROUP_M * tiles_n) * GROUP_M
    size = min(tiles_m - first, GROUP_M)
    r = pid % (GROUP_M * tiles_n)
    return first + r % size, r // size


def moe_find(off, E, T, tile, cap, tiles_n, bid, lanes=64):
    """Restatement of the kernel's lookup with `lanes` lanes: every lane counts its consecutive experts, the first
    whose saturating prefix sum passes the m-tile owns it, and a second pass finds the expert among its own.
    Returns (expert, m-tile of the expert, n-tile, first row, rows), or None past the last tile."""
    def count(e):
        lo = min(max(int(off[min(e, E)]), 0), T)
        hi = min(max(int(off[min(e + 1, E)]), lo), T)
        return lo, hi, -(-(hi - lo) // tile)

    def prefix(ns):
        out, s = [], 0
        for n in ns:
            s = min(s + n, cap)
            out.append(s)
        return out

    def owner(incl, mt):
        lane = next(i for i, s in enumerate(incl) if s > mt)
        return lane, mt - (incl[lane - 1] if lane else 0)

    per = -(-E // lanes)
    incl = prefix([min(sum(count(lane * per + k)[2] for k in range(per)), cap) for lane in range(lanes)])
    total = incl[-1]
    if bid >= total * tiles_n:
        return None
    mt, tn = tile_coords(bid, total * tiles_n, total, tiles_n)
    lane, mt = owner(incl, mt)
    e = lane * per
    for k in range(0, per, lanes) if per > 1 else ():
        incl = prefix([min(count(e + k + i)[2], cap) if k + i < per else 0 for i in range(lanes)])
        if mt < incl[-1]:
            lane, mt = owner(incl, mt)
            e += k + lane
            break
        mt -= incl[-1]
    else:
        assert per == 1
    lo, hi, _ = count(e)
    return e, mt, tn, lo, hi - lo


# (experts, lanes): one expert per lane, several, and more than one pass over a lane's own.
LOOKUPS = [(1, 64), (20, 64), (64, 64), (65, 64), (70, 64), (300, 64), (30, 4), (90, 4)]


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("E,lanes", LOOKUPS)
def test_moe_lookup_covers_valid_tables_exactly_once(E, lanes, tile):
    """Every workgroup of the grid that has a tile has its own, and together they are the experts' rows."""
    rng = np.random.default_rng(E * tile)
    for mean, tiles_n in ((3, 2), (tile, 1), (2 * tile, 3)):
        counts = rng.integers(0, 2 * min(mean, 60_000 // E) + 1, E)
        counts[rng.random(E) < 0.3] = 0
        off = np.concatenate([[0], np.cumsum(counts)])
        T = int(off[-1]) + int(rng.integers(0, 300))
        bound = grid_m(T, E, tile)
        seen, rows = set(), np.zeros(T, dtype=int)
        real = int(np.sum(-(-counts // tile)))
        assert real <= bound
        bids = range(bound * tiles_n) if real <= 300 else sorted(rng.choice(bound * tiles_n, 300, replace=False))
        for bid in bids:
            r = moe_find(off, E, T, tile, bound, tiles_n, int(bid), lanes)
            assert (r is None) == (bid >= real * tiles_n)
            if r is None:
                continue
            e, mt, tn, lo, n = r
            assert lo == off[e] and n == counts[e] and 0 <= mt < -(-n // tile) and 0 <= tn < tiles_n
            assert (e, mt, tn) not in seen
            seen.add((e, mt, tn))
            rows[lo + tile * mt:lo + min(tile * (mt + 1), n)] += tn == 0
        if len(bids) == bound * tiles_n:
            assert len(seen) == real * tiles_n
            assert np.all(rows[:off[-1]] == 1) and np.all(rows[off[-1]:] == 0)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("E,lanes", LOOKUPS)
def test_moe_lookup_keeps_garbage_tables_in_bounds(E, lanes, tile):
    rng = np.random.default_rng(E + tile)
    for _ in range(6):
        T = int(rng.integers(1, 3000))
        off = rng.integers(-5000, 8000, E + 1)
        bound = grid_m(T, E, tile)
        for bid in rng.integers(0, bound * 2, 60):
            r = moe_find(off, E, T, tile, bound, 2, int(bid), lanes)
            if r is None:
                continue
            e, mt, tn, lo, rows = r
            assert 0 <= e < E and 0 <= tn < 2 and 0 <= lo and lo + rows <= T
            # rows the tile reads from A and writes to C
            first, last = lo + tile * mt, lo + min(tile * (mt + 1), rows)
            assert 0 <= first < last <= T
