"""How a large matmul is split over the int8 path's scratch (csrc/gemm.hip, gemm_split.hip): host decisions, no GPU.

A call that does not fit the scratch runs in row blocks that share B's split, which the first block makes. So either all
of a call's blocks run on the int8 path or none, and only the first is without a split to take."""

from __future__ import annotations

import ctypes as C
import random

import pytest

import matmul_calls as M

pytestmark = pytest.mark.skipif(not M.HARNESS.exists(), reason="tests/native is not built")

GIB = 1 << 30
# calls whose full blocks, asked one by one, are quicker on FP64 while the smaller last block is not (its tiles fill the
# last round of workgroups better): a head's input gradient, its forward and its windowed weight gradient, two layers'
UNEVEN = [
    M.row_major(33304, 256, 32000, cap=2 * GIB),
    M.row_major(2308, 256000, 576, cap=GIB),
    M.windowed(151936, 1536, 4600, 8, 575, cap=5 * GIB),
    M.row_major(2912, 1452, 2888, cap=66501847),
    M.windowed(2832, 1512, 5282, 6, 3169, cap=241863356),
]


def assert_blocks(h, call: M.MatmulCall):
    made = M.blocks(h, call)
    rows = h.matmul_rows(C.byref(call))
    what = (call.I, call.J, call.L, call.nseg, call.cap, made)
    if not rows:
        return made
    assert sum(b[0] for b in made) == call.I and all(b[0] == rows for b in made[:-1]), what
    assert all(on_int8 == n for n, on_int8, _ in made), what
    assert [ready for _, _, ready in made] == [0] + [1] * (len(made) - 1), what
    return made


@pytest.mark.parametrize("call", UNEVEN, ids=lambda c: f"{c.I}x{c.J}x{c.L}")
def test_blocks_whose_last_alone_would_pay(call):
    h = M.load()
    made = assert_blocks(h, call)
    assert len(made) > 1 and made[-1][0] < made[0][0]


def test_blocks_of_any_call_and_scratch():
    h, rng, several = M.load(), random.Random(7), 0
    for _ in range(20000):
        rows, cols, length = (int(2 ** rng.uniform(8, 17)) // 4 * 4 for _ in range(3))
        nseg = rng.choice([0, 1, 2, 8, 64])
        call = M.row_major(rows, cols, length) if rng.random() < 0.5 else \
            M.windowed(rows, cols, length, nseg, min(length, 2 * length // max(nseg, 1)))
        call.cap = int(h.matmul_bytes(C.byref(call)) * rng.uniform(0.05, 1.1))
        several += len(assert_blocks(h, call)) > 1
    assert several > 1000  # the sweep reaches what it is about


# measured: a call, the tiles it handed back and the outputs it recomputed, its milliseconds on the int8 path and on FP64
MEASURED = [
    (M.windowed(151936, 1536, 8192, 8, 1024, cap=5 * GIB), 0, 689183, 47.8, 55.5),  # the logits' gradient: flat logits ...
    (M.windowed(151936, 1536, 8192, 8, 1024, cap=5 * GIB), 0, 2383861, 53.1, 55.4),
    (M.windowed(151936, 1536, 8192, 8, 1024, cap=5 * GIB), 0, 3414249, 73.6, 55.5),
    (M.windowed(151936, 1536, 8192, 8, 1024, cap=5 * GIB), 0, 4395842, 112.9, 55.4),  # ... to peaked ones
    (M.windowed(50304, 2048, 8192, 4, 2048), 0, 243911, 18.0, 24.4),
    (M.windowed(50304, 2048, 8192, 4, 2048), 0, 1967082, 48.3, 24.3),
    (M.windowed(32768, 1536, 8192, 8, 1024), 0, 990948, 25.3, 11.9),
    (M.windowed(65536, 1024, 2048, 2, 1024), 0, 343055, 6.2, 4.0),
    (M.row_major(1918, 1056, 3232), 0, 12000, 0.265, 0.244),  # an MLP's product through its down projection
    (M.row_major(8192, 1536, 8960), 0, 57000, 3.05, 3.77),
    (M.row_major(8192, 1536, 151936, cap=5 * GIB), 100, 24000, 78.0, 58.0),  # a few handed-back tiles of a long reduction
    (M.row_major(1030, 1792, 36000), 150, 16384, 4.2, 2.6),
]


@pytest.mark.parametrize("call,tiles,chains,int8,fp64", MEASURED, ids=lambda v: f"{v.I}x{v.J}x{v.L}" if hasattr(v, "I") else None)
def test_recomputation_that_costs_more_than_the_path_saves(call, tiles, chains, int8, fp64):
    h = M.load()
    assert h.matmul_rows(C.byref(call)) > 0
    assert bool(h.matmul_lost(C.byref(call), tiles, chains)) == (int8 > fp64)
