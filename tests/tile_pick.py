"""The library's choice of the output tile (csrc/g9_tile_pick.hpp, host code),
compiled with the host compiler and called for given sizes on 256 CUs."""

import ctypes
import functools
import os
import subprocess
import tempfile

from gfx950_gluon_tutorials_amd import _lib

HEADER = os.path.join(os.path.dirname(_lib.__file__), "csrc", "g9_tile_pick.hpp")
CUS = 256
# Operand kind: (cost family, bytes per value, values per K stage)
KINDS = {"f16": (0, 2.0, 64), "bf16": (0, 2.0, 64), "bf8": (1, 1.0, 128), "mxfp4": (2, 0.53125, 256)}

_SOURCE = f"""
#include "{HEADER}"
using namespace g9;
extern "C" void tile_of(int shape, int* out) {{ out[0] = kTileShapes[shape][0]; out[1] = kTileShapes[shape][1]; }}
extern "C" int dense(int family, long long M, long long N, int ns, double bytes, long long lda, long long ldsa) {{
  return pick_tile(TileProblem{{family, M, N, ns, bytes, lda, ldsa, {CUS}}});
}}
extern "C" int beats(int family, long long M, long long N, int ns, double bytes, long long lda, int shape,
                     long long tiles, int S, int ragged) {{
  return tile_beats_split(TileProblem{{family, M, N, ns, bytes, lda, 0, {CUS}}}, shape, tiles, S, ragged);
}}
extern "C" int moe(int family, long long T, long long E, long long N, int ns, double bytes, long long lda) {{
  return pick_moe_tile(TileProblem{{family, T, N, ns, bytes, lda, 0, {CUS}}}, E);
}}
"""


@functools.cache
def _pick():
    with tempfile.TemporaryDirectory(prefix="g9pick") as d:
        src, so = os.path.join(d, "pick.cpp"), os.path.join(d, "pick.so")
        with open(src, "w") as fh:
            fh.write(_SOURCE)
        subprocess.run(["g++", "-std=c++20", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", src, "-o", so], check=True)
        lib = ctypes.CDLL(so)
    i, q, f = ctypes.c_int, ctypes.c_longlong, ctypes.c_double
    lib.dense.argtypes = [i, q, q, i, f, q, q]
    lib.beats.argtypes = [i, q, q, i, f, q, i, q, i, i]
    lib.moe.argtypes = [i, q, q, q, i, f, q]
    return lib


def _tile(shape):
    out = (ctypes.c_int * 2)()
    _pick().tile_of(shape, out)
    return f"{out[0]}x{out[1]}"


def _row(kind, K):
    """Bytes of a packed operand row."""
    return K // 2 if kind == "mxfp4" else int(K * KINDS[kind][1])


def dense(kind, M, N, K, lda=None):
    """The tile of a data-parallel launch, as "<rows>x<columns>"."""
    family, value, stage = KINDS[kind]
    lda = _row(kind, K) if lda is None else lda
    return _tile(_pick().dense(family, M, N, -(-K // stage), (M + N) * K * value + 2 * M * N, lda, 0))


def factor(kind, M, N, K):
    """Split-K's segments per 256x256 tile where it splits."""
    return _lib.load().g9_splitk_factor(-(-M // 256) * -(-N // 256), -(-K // KINDS[kind][2]), CUS)


def splitk(kind, M, N, K, lda=None, off_line=False):
    """The segments per 256x256 tile of a split-K call, or the tile of the data-parallel launch it becomes; off_line:
    the operands start off a 128-byte line."""
    family, value, stage = KINDS[kind]
    row = _row(kind, K)
    lda = row if lda is None else lda
    tiles, ns = -(-M // 256) * -(-N // 256), -(-K // stage)
    S = factor(kind, M, N, K)
    bytes_ = (M + N) * K * value + 2 * M * N
    shape = _pick().dense(family, M, N, ns, bytes_, lda, 0)
    ragged = off_line or lda % 128 != 0 or row % 128 != 0  # (row: a K tail shifts every stage)
    if S <= 1 or _pick().beats(family, M, N, ns, bytes_, lda, shape, tiles, S, ragged):
        return _tile(shape)
    return S


def moe(kind, T, E, N, K):
    """The tile of a grouped launch of T rows over E experts."""
    family, value, stage = KINDS[kind]
    bytes_ = (T + min(E, T) * N) * K * value + 2 * T * N
    return _tile(_pick().moe(family, T, E, N, -(-K // stage), bytes_, _row(kind, K)))
