"""CPU checks of the rules that choose between small tiles, 256x256 tiles and
split-K: what they pick where both sides were measured, and that no tile is
picked that cannot address its operands."""

import random

import pytest

import tile_pick as P

# (operands, M, N, K): small tile, or the split, by measurement on one MI355X
# (256 CUs): us per call of the tile and of the split, operands in the
# memory-side cache / from HBM.
SPLIT_RULE = [
    (("f16", 512, 4096, 8192), "128x64"),        # 37.3 / 53.4, 47.3 / 48.1
    (("f16", 227, 7526, 3904), "128x64"),        # 21.8 / 30.4, 35.1 / 37.4
    (("bf16", 1, 5043, 23744), "16x32"),         # 42.5 / 42.4, 67.6 / 67.0
    (("bf16", 865, 8039, 9984), 2),              # 150, 137.6
    (("bf8", 1874, 3840, 5760), "256x128"),      # 35.1 / 44.3, 50.8 / 51.8
    (("bf8", 7972, 896, 22272), 2),              # 159.4 / 158.7, 121.6 / 122.1
    (("bf8", 120, 4763, 23040), 13),             # 56.0, 42.3
    (("bf8", 5275, 512, 17616), 6),              # rows off 128-byte lines: 85.4, 57.0
    (("mxfp4", 1016, 3584, 18176), "128x128"),   # 38.9 / 49.5, 49.8 / 51.0
    (("mxfp4", 281, 7936, 32000), 4),            # 83.5, 66.4
    (("mxfp4", 639, 8184, 28928), 2),            # 102.6 / 119.9, 95.0 / 96.7
]


@pytest.mark.parametrize("problem,want", SPLIT_RULE)
def test_splitk_calls_take_the_faster_side(problem, want):
    assert P.splitk(*problem) == want


# Rows whole lines apart, but stages off them by the base (K whole lines) or by a K tail: us of the tile and of the split.
OFF_LINES = [(("bf16", 1731, 664, 6080), 12),     # 47.2, 35.7
             (("bf8", 4174, 368, 14080), 7),      # 57.1, 43.2
             (("bf16", 354, 4144, 9448), 7),      # 69.6, 47.8
             (("bf8", 5169, 384, 19744), 6)]      # 80.9, 56.6


@pytest.mark.parametrize("problem,want", OFF_LINES)
def test_stages_off_lines_stay_split(problem, want):
    kind, K = problem[0], problem[3]
    lda = -(-P._row(kind, K) // 128) * 128
    assert P.splitk(*problem, lda=lda, off_line=True) == want
    assert (P.splitk(*problem, lda=lda) == want) == (lda != P._row(kind, K))


@pytest.mark.parametrize("kind", list(P.KINDS))
def test_tiles_address_their_rows(kind):
    """From row strides of 2^23 bytes on the 256-row tile is no choice, and the next best one is
    taken: a split-K call never leaves the split for 256x256 tiles."""
    rng = random.Random(0)
    wide = 0
    for _ in range(400):
        M, N, K = rng.randint(300, 8000), rng.randint(300, 8000), rng.randint(1, 40) * 256
        near, far = P.dense(kind, M, N, K), P.dense(kind, M, N, K, lda=2**23)
        assert far != "256x128" and (near == far or near == "256x128")
        wide += near == "256x128"
        s = P.splitk(kind, M, N, K, lda=2**23)
        assert s != "256x256" or P.factor(kind, M, N, K) == 1
    assert wide > 10
