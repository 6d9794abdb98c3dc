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
