"""ctypes side of tests/native/matmul_calls.cpp: the library's internal matmul call for the tests."""

from __future__ import annotations

import ctypes as C
from pathlib import Path

HARNESS = Path(__file__).resolve().parent / "native" / "libmatmul_calls.so"

_P, _N = C.c_void_p, C.c_int64


class MatmulCall(C.Structure):
    _fields_ = ([(n, _P) for n in ("A", "B", "Bt", "C")] +
                [(n, _N) for n in ("a_kind", "lda", "ldb", "ldbt", "ldc", "I", "J", "L")] +
                [("seg", _P), ("nseg", _N), ("seg_max", _N)] +
                [(n, _P) for n in ("bias", "addsrc", "addrow", "addend", "weight", "rowscale", "partial")] +
                [("partial_cap", _N), ("scratch", _P), ("cap", _N), ("bt_transpose", _P), ("share", _N), ("ready", _N),
                 ("stat", _P)])


def load(path: Path = HARNESS) -> C.CDLL:
    h = C.CDLL(str(path))
    for name in ("matmul_rows", "matmul_bytes", "matmul_blocks"):
        getattr(h, name).restype = _N
    h.matmul_blocks.argtypes = [C.POINTER(MatmulCall), _N] + [C.POINTER(_N)] * 3
    h.matmul_lost.argtypes = [C.POINTER(MatmulCall), C.c_uint32, C.c_uint32]
    h.matmul_run.argtypes = [C.POINTER(MatmulCall), _P]
    return h


SOMEWHERE = 1 << 20  # an aligned address, for calls that are only planned


def row_major(rows: int, cols: int, length: int, *, b_t: bool = True, **more) -> MatmulCall:
    """out[rows][cols] = x[rows][length] times B, given as [length][cols] and, with b_t, as [cols][length] too."""
    return MatmulCall(**{**dict(A=SOMEWHERE, B=SOMEWHERE, Bt=SOMEWHERE if b_t else None, C=SOMEWHERE, a_kind=2, lda=length,
                                ldb=cols, ldbt=length, ldc=cols, I=rows, J=cols, L=length, nseg=1, scratch=SOMEWHERE,
                                cap=1 << 62), **more})


def windowed(rows: int, cols: int, length: int, nseg: int = 0, longest: int = 0, **more) -> MatmulCall:
    """out[rows][cols] = the sum over nseg windows of dy[length][rows]^T x[length][cols] (nseg 0: one plain reduction)."""
    return MatmulCall(**{**dict(A=SOMEWHERE, B=SOMEWHERE, C=SOMEWHERE, a_kind=1, lda=rows, ldb=cols, ldc=cols, I=rows,
                                J=cols, L=length, seg=SOMEWHERE if nseg else None, nseg=max(nseg, 1), seg_max=longest,
                                scratch=SOMEWHERE, cap=1 << 62), **more})


def blocks(h: C.CDLL, call: MatmulCall, most: int = 4096):
    """The call's row blocks on the int8 path: (rows, rows on that path, takes B's split as made) of each."""
    out = [(_N * most)() for _ in range(3)]
    n = h.matmul_blocks(C.byref(call), most, *out)
    return [tuple(int(o[k]) for o in out) for k in range(n)]
