"""What a prepared GEMM launch runs, read from its plan: the words of struct
Plan (csrc/g9_capi.hip) hold the grid and the reduction's grid, which is 0 for
anything but split-K.  The wrappers resolve their launches the same way."""

import ctypes

from gfx950_gluon_tutorials_amd.gemm.prepared import PreparedGemm


def _check(prep: PreparedGemm, M: int, N: int, want) -> None:
    words = (ctypes.c_uint32 * 5).from_buffer(prep._plans[0])
    grid, reduction = words[2], words[4]
    if isinstance(want, int):
        assert reduction and grid == -(-M // 256) * -(-N // 256) * want, f"grid {grid} is not {want} segments a tile"
    else:
        tm, tn = map(int, want.split("x"))
        assert not reduction and grid == -(-M // tm) * -(-N // tn), f"grid {grid} is not of {want} tiles"


def a16w16(want, a, b_kn, c, **kw):
    """Asserts that the call launches `want`: a tile ("128x64"), or split-K's segments per 256x256 tile."""
    _check(PreparedGemm.a16w16([(a, b_kn, c)], **kw), a.shape[0], b_kn.shape[1], want)


def a8w8(want, a, b_kn, c, sa=None, sb=None, **kw):
    _check(PreparedGemm.a8w8([(a, b_kn, c, sa, sb)], **kw), a.shape[0], b_kn.shape[1], want)


def a4w4(want, a, b, sa, sb, c, **kw):
    _check(PreparedGemm.a4w4([(a, b, sa, sb, c)], **kw), a.shape[0], b.shape[0], want)
