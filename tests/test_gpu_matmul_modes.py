"""GPU parity of the int8 matmul path's modes that only the trainer reaches (csrc/gemm_split.hip): whole outputs against
the same call without scratch, which runs on FP64 (each output's bits do not depend on the path), and a few of them against
serial double sums. Operands with ordinary and very wide rows, exact ties, zero rows, infinities and NaNs; sizes off the
path's tiles and steps; a scratch that holds other bytes before."""

from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import matmul_calls as M
from test_gpu_split_matmul import KINDS, assert_same, operand

pytestmark = pytest.mark.gpu


class Call:
    """One matmul call over device copies of its operands (extra: further operands and fields, by MatmulCall's names)."""

    def __init__(self, plan: M.MatmulCall, a: np.ndarray, b: np.ndarray, **extra):
        from etalii_dllm_amd import kernels as K

        self.K, self.h, self.m, self.keep = K, M.load(), plan, []
        plan.A, plan.B = self.up(a), self.up(b)
        if plan.Bt:
            plan.Bt = self.up(b.T)
        for name, value in extra.items():
            setattr(plan, name, self.up(value) if isinstance(value, np.ndarray) else value)
        if plan.partial:
            plan.partial = self.new(4 * plan.partial_cap)
        self.out_bytes = 4 * plan.I * plan.J
        if plan.cap >= 1 << 62:
            plan.cap = self.h.matmul_bytes(C.byref(plan))
        self.scratch = self.new(plan.cap, 0x5a)
        plan.stat = self.new(8)

    def up(self, x: np.ndarray) -> int:
        self.keep.append(self.K.Device.of(x))
        return self.keep[-1].ptr.value

    def new(self, nbytes: int, fill: int = 0) -> int:
        self.keep.append(self.K.Device(nbytes))
        self.K.check(self.K.lib.dllm_hip_memset(self.keep[-1].ptr, fill, nbytes))
        return self.keep[-1].ptr.value

    def rows(self) -> int:
        """Rows per block on the int8 path."""
        self.m.scratch = self.scratch
        return self.h.matmul_rows(C.byref(self.m))

    def redone(self) -> tuple[int, int]:
        """Tiles handed back to FP64 and outputs recomputed by their chains, so far."""
        out = np.empty(2, np.uint32)
        self.K.check(self.K.lib.dllm_hip_download(out.ctypes.data, self.m.stat, 8))
        return int(out[0]), int(out[1])

    def run(self, int8: bool, seed: np.ndarray | None = None) -> np.ndarray:
        """The call's output, on the int8 path or on FP64; seed: what the output holds before, and the addend."""
        out = self.K.Device(self.out_bytes)
        self.K.check(self.K.lib.dllm_hip_memset(out.ptr, 0x7f, self.out_bytes))
        if seed is not None:
            self.K.check(self.K.lib.dllm_hip_upload(out.ptr, np.ascontiguousarray(seed).ctypes.data, self.out_bytes))
            self.m.addsrc = out.ptr.value
        self.m.C, self.m.scratch = out.ptr.value, self.scratch if int8 else None
        self.K.check(self.h.matmul_run(C.byref(self.m), None))
        return out.download((self.m.I, self.m.J))


def chain(a: np.ndarray, b: np.ndarray) -> float:
    """The serial double sum of float products (exact in double, so each addition rounds once)."""
    with np.errstate(all="ignore"):
        return float(np.add.accumulate(a.astype(np.float64) * b.astype(np.float64))[-1]) if len(a) else 0.0


@pytest.mark.parametrize("kind", KINDS)
def test_row_blocks(kind):
    """Blocks of 1536 and 1376 rows that share B's split, with a bias and onto an addend in place. Asked by itself the
    first block would be left to FP64."""
    rows, cols, length = 2912, 1452, 2888
    x, w = operand(kind, 1, rows, length), operand("gauss" if kind == "special" else kind, 2, cols, length)
    bias, onto = operand("gauss", 3, 1, cols)[0], operand("gauss", 4, rows, cols)
    c = Call(M.row_major(rows, cols, length, cap=66501847), x, w.T, bias=bias)
    assert c.rows() == 1536
    got, want = c.run(True, onto), c.run(False, onto)
    assert_same(got, want, kind)
    for i, j in ((0, 0), (1535, 5), (1536, cols - 1), (rows - 1, 77)):
        with np.errstate(all="ignore"):
            exact = onto[i, j] + np.float32(chain(x[i], w[j]) + float(bias[j]))
        assert_same(got[i:i + 1, j], np.array([exact], np.float32), f"{kind} {i} {j}")


def windows_of(length: int) -> np.ndarray:
    """Six windows of a reduction: empty ones, one row, one below a step, two long ones."""
    sizes = [0, 1, length // 2 - 7, 63, 0]
    return np.cumsum([0] + sizes + [length - sum(sizes)]).astype(np.int64)


def weight_gradient(kind: str, rows: int, cols: int, length: int, **plan):
    """A windowed call with addends, row factors and window factors; its operands and their host copies."""
    seg = windows_of(length)
    dy, x = operand(kind, 5, length, rows), operand("gauss" if kind == "special" else kind, 6, length, cols)
    rng = np.random.default_rng(8)
    addrow = rng.integers(-1, 40, (6, rows)).astype(np.int32)
    addend, rowscale = operand("gauss", 9, 40, cols), operand("gauss", 10, 1, rows)[0]
    weight = operand("gauss", 11, 1, 6)[0]
    c = Call(M.windowed(rows, cols, length, 6, int(np.diff(seg).max()), **plan), dy, x, seg=seg, addrow=addrow,
             addend=addend, rowscale=rowscale, weight=weight)

    def exact(i: int, j: int) -> np.float32:
        total = np.float32(0.0)
        with np.errstate(all="ignore"):
            for s in range(6):
                v = np.float32(chain(dy[seg[s]:seg[s + 1], i], x[seg[s]:seg[s + 1], j]))
                v = v + (addend[addrow[s, i], j] if addrow[s, i] >= 0 else np.float32(0.0))
                v = v * rowscale[i] * weight[s]
                total = v if s == 0 else total + v
        return total

    return c, exact


def check(c: Call, exact, picks, kind: str) -> None:
    got, want = c.run(True), c.run(False)
    assert_same(got, want, kind)
    for i, j in picks:
        assert_same(got[i:i + 1, j], np.array([exact(i, j)], np.float32), f"{kind} {i} {j}")
    tiles, chains = c.redone()
    assert (tiles == 0 and chains > 0) if kind == "gauss" else tiles + chains > 0


@pytest.mark.parametrize("kind", KINDS)
def test_windows_in_sequence(kind):
    c, exact = weight_gradient(kind, 1516, 1344, 5224)
    assert c.rows() == 1516 and not c.h.matmul_parallel(C.byref(c.m))
    check(c, exact, ((0, 0), (70, 11), (131, 700), (1515, 1343)), kind)


@pytest.mark.parametrize("kind", KINDS)
def test_windows_in_parallel(kind):
    c, exact = weight_gradient(kind, 1836, 648, 3458, partial=1, partial_cap=6 * 1836 * 648)
    assert c.rows() == 1836 and c.h.matmul_parallel(C.byref(c.m))
    check(c, exact, ((0, 0), (70, 11), (131, 500), (1835, 647)), kind)


@pytest.mark.parametrize("kind", KINDS)
def test_row_blocks_of_windows(kind):
    c, exact = weight_gradient(kind, 2832, 1512, 5282, cap=241863356)
    assert c.rows() == 1536
    check(c, exact, ((0, 0), (1535, 11), (1536, 700), (2831, 1511)), kind)


def softmax_gradient(seed: int, rows: int, cols: int, spread: float) -> np.ndarray:
    """Rows of a cross-entropy's gradient: a softmax (of logits of this deviation) less one at the target."""
    p = np.exp(spread * operand("gauss", seed, rows, cols))
    p /= p.sum(axis=1, keepdims=True)
    p[np.arange(rows), np.random.default_rng(seed).integers(0, cols, rows)] -= np.float32(1.0)
    return (p / np.float32(rows)).astype(np.float32)


@pytest.mark.parametrize("kind,length", [(k, 21856) for k in KINDS] + [("flat", 21856), ("flat", 43652), ("peaked", 21856)])
def test_long_reduction(kind, length):
    """Legs of 21824 l, the last one short, and rows with one value far above the others kept apart. (A peaked softmax spans
    too many digits: all its tiles come back to FP64.)"""
    rows, cols = 1420, 988
    spread = {"flat": 0.5, "peaked": 2.0}.get(kind)
    dy = softmax_gradient(12, rows, length, spread) if spread else operand(kind, 12, rows, length)
    w = operand("gauss" if kind == "special" or spread else kind, 13, length, cols)
    onto = operand("gauss", 14, rows, cols)
    c = Call(M.row_major(rows, cols, length), dy, w)
    assert c.rows() == rows
    got, want = c.run(True, onto), c.run(False, onto)
    assert_same(got, want, kind)
    for i, j in ((0, 0), (3, 5), (70, 9), (131, 987), (1419, 400)):
        with np.errstate(all="ignore"):
            exact = onto[i, j] + np.float32(chain(dy[i], w[:, j]))
        assert_same(got[i:i + 1, j], np.array([exact], np.float32), f"{kind} {i} {j}")
    tiles, chains = c.redone()
    assert (tiles == 0 and chains > 0) if kind in ("gauss", "flat") else tiles + chains > 0


@pytest.mark.parametrize("kind", KINDS)
def test_calls_that_share_their_rows(kind):
    """Two projections of the same rows and, between them, one that the path does not take: the rows are split once, for
    both widths."""
    rows, length = 2049, 1540
    x = operand(kind, 15, rows, length)
    w = [operand("gauss", 16 + k, n, length) for k, n in enumerate((2236, 40, 3284))]
    calls = [Call(M.row_major(rows, len(v), length, cap=1 << 30), x, v.T) for v in w]
    for k, c in enumerate(calls):
        c.m.A, c.scratch, c.m.share, c.m.ready = calls[0].m.A, calls[0].scratch, 1, k > 0
    assert [c.rows() for c in calls] == [rows, 0, rows]
    got = [c.run(True) for c in calls]
    for c, g in zip(calls, got):
        assert_same(g, c.run(False), kind)
