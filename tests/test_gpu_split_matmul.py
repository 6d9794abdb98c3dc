"""GPU parity of the matmuls' int8 matrix-core path (csrc/gemm_split.hip): whole outputs against the same calls in pieces
too small for that path (each output's bits do not depend on the call around it), and sampled rows against the oracle,
bit for bit. Sizes off the path's 64 x 64 tiles, 64-l steps and 256-l parts; operands with ordinary and very wide rows,
exact ties, zero rows, infinities and NaNs, so that every way an output is decided is taken."""

from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import matmul_calls as M
import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from etalii_dllm_amd import kernels

    return kernels


def operand(kind: str, seed: int, rows: int, cols: int) -> np.ndarray:
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((rows, cols)).astype(np.float32)
    if kind == "tail":  # a few bits per row lost below the sixth digit
        x = x * np.exp(1.5 * rng.standard_normal((rows, cols))).astype(np.float32)
    elif kind == "wide":  # rows and columns of very different size, and values from 1e-30 to 1e10 inside some
        x = x * np.power(10.0, rng.integers(-12, 9, (rows, 1))).astype(np.float32)
        x[::5] *= np.power(10.0, rng.integers(-18, 2, (len(x[::5]), cols))).astype(np.float32)
    elif kind == "ties":  # sums that are small integers: exact zeros, ties of the rounding
        x = rng.integers(-3, 4, (rows, cols)).astype(np.float32)
        x[:, 0] = 4096.0 * rng.integers(-1024, 1025, rows)
        x[::3, 1] = 2.0 ** -12
    elif kind == "special":
        x[3] = 0.0
        x[:, 5] = 0.0
        x[70, 11], x[71, 12], x[200, 13] = np.inf, -np.inf, np.nan
        x[130] = np.float32(1e-42) * x[130]
        x[131] = np.float32(3e37) * np.sign(x[131])
    return np.ascontiguousarray(x)


KINDS = ["gauss", "tail", "wide", "ties", "special"]


def assert_same(a: np.ndarray, b: np.ndarray, what: str) -> None:
    nan = np.isnan(a) & np.isnan(b)
    bad = (a.view(np.uint32) != b.view(np.uint32)) & ~nan
    assert not bad.any(), (what, int(bad.sum()), a.size, np.argwhere(bad)[:4].tolist())


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("rows,inf,outf,int8", [(2049, 1540, 4868, True), (1300, 8196, 1348, True), (4100, 644, 5444, True),
                                                (1000, 8196, 1348, False), (4100, 516, 5444, False)])
def test_linear(K, kind, rows, inf, outf, int8):
    """int8: which path the whole call takes (the pieces are all FP64's)."""
    h = M.load()
    assert bool(h.matmul_rows(C.byref(M.row_major(rows, outf, inf)))) == int8
    assert not h.matmul_rows(C.byref(M.row_major(256, 512, inf)))
    x, w = operand(kind, 1, rows, inf), operand("gauss" if kind == "special" else kind, 2, outf, inf)
    b = operand("gauss", 3, 1, outf)[0]
    got = K.linear(x, w, b)
    parts = [K.linear(x[i:i + 256], w[j:j + 512], b[j:j + 512]) for i in range(0, rows, 256)
             for j in range(0, outf, 512)]
    nj = -(-outf // 512)
    want = np.concatenate([np.concatenate(parts[k * nj:(k + 1) * nj], axis=1) for k in range(-(-rows // 256))])
    assert_same(got, want, "linear")
    pick = np.array([0, 3, 70, 130, 131, rows - 1])
    assert_same(got[pick][:, -70:], O.oracle_kernels().linear(x[pick], w[-70:].copy(), b[-70:].copy()), "oracle")


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("rows,inf,outf", [(2051, 900, 4868), (8191, 1028, 1540)])
def test_linear_backward(K, kind, rows, inf, outf):
    h = M.load()
    assert h.matmul_rows(C.byref(M.row_major(rows, inf, outf, b_t=False))) and h.matmul_rows(C.byref(M.windowed(outf, inf, rows)))
    assert not h.matmul_rows(C.byref(M.row_major(128, inf, outf, b_t=False)))
    assert not h.matmul_rows(C.byref(M.windowed(128, inf, rows)))
    x, w = operand("gauss", 4, rows, inf), operand("gauss", 5, outf, inf)
    dy = operand(kind, 6, rows, outf)
    dx, dw, db = K.linear_backward(x, w, dy, with_bias=True)
    want = np.concatenate([K.linear_backward(x[i:i + 128], w, dy[i:i + 128])[0] for i in range(0, rows, 128)])
    assert_same(dx, want, "dx")
    pieces = [K.linear_backward(x, w[j:j + 128], np.ascontiguousarray(dy[:, j:j + 128]), with_bias=True)
              for j in range(0, outf, 128)]
    assert_same(dw, np.concatenate([p[1] for p in pieces]), "dw")
    assert_same(db, np.concatenate([p[2] for p in pieces]), "db")
    cols = np.array([0, 11, 12, outf - 1])
    ora = O.oracle_kernels().linear_backward(x, w[cols].copy(), dy[:, cols].copy())
    assert_same(dw[cols], ora[1], "oracle dw")


@pytest.mark.parametrize("kind", ["gauss", "wide", "special"])
@pytest.mark.parametrize("rows,inf,outf", [(1, 132, 36), (1, 896, 4864), (2, 1028, 4092), (5, 252, 1000), (1, 4, 40)])
def test_linear_of_few_rows(K, kind, rows, inf, outf):
    """A token or a few through a projection: every output by its own chain."""
    x, w = operand("gauss", 7, rows, inf), operand(kind if inf > 13 and outf > 200 else "gauss", 8, outf, inf)
    b = operand("gauss", 9, 1, outf)[0]
    assert_same(K.linear(x, w, b), O.oracle_kernels().linear(x, w, b), "linear")
    assert_same(K.linear(x, w), K.linear(np.repeat(x, 80, axis=0), w)[::80], "the same rows in a larger call")


@pytest.mark.parametrize("other_rows,hot_rows", [(False, 2048), (True, 2048), (False, 512)])
def test_a_resting_matmul_runs_grouped_and_comes_back(other_rows, hot_rows):
    """A layer's gate and up projections hand the tiles of hot_rows rows back once (a channel of great size meets zero
    weights, so the results lie far below the operands' digits), which costs more than the path saves. They rest for 32
    steps as one grouped FP64 launch, and return to the int8 path as two calls, whatever row counts the steps between had.
    Counted by the matmul launches of a step."""
    from etalii_dllm_amd import kernels
    from etalii_dllm_amd.trainer import Decoder, Trainer

    lib = kernels.lib
    h = M.load()
    for n in (2048, 2044):  # of the layer's matmuls gate, up and down's input gradient are the int8 path's
        assert h.matmul_rows(C.byref(M.row_major(n, 3712, 896))) == n
        assert not any(h.matmul_rows(C.byref(M.row_major(n, *s))) for s in ((896, 3712), (896, 896)))
    t = Trainer(Decoder(256, 896, 3712, 1, 14, 2, 64, 1e-6, 1e4, True), 2048, 2, 1024)
    rng = np.random.default_rng(3)
    dims = {"token_embedding": (256, 896), "q": (896, 896), "k": (128, 896), "v": (128, 896), "o": (896, 896),
            "gate": (3712, 896), "up": (3712, 896), "down": (896, 3712)}
    weights = {n: np.ones(896, np.float32) if n.endswith("norm.weight") else
               (0.02 * rng.standard_normal(dims[n.split(".")[-2]])).astype(np.float32) for n in t.names}
    for name in ("gate", "up"):
        weights[f"layers.0.mlp.{name}.weight"][:, 0] = 0.0
    weights["layers.0.attention.o.weight"][0] = 0.0  # the channel is the embedding's: tokens of 128 and above have none
    weights["token_embedding.weight"][128:, 0] = 0.0
    hot = {**weights, "layers.0.mlp_norm.weight": weights["layers.0.mlp_norm.weight"].copy()}
    hot["layers.0.mlp_norm.weight"][0] = 1e9
    tokens = np.concatenate([rng.integers(0, 128, hot_rows), rng.integers(128, 256, 2049 - hot_rows)]).tolist()
    windows = {n: [tokens[:1025], tokens[1024:n + 1]] for n in (2048, 2044)}
    step = 0

    def launches(rows: int) -> tuple[int, int]:
        """A step's matmul launches, and those of them on the int8 path."""
        nonlocal step
        step += 1
        kernels.check(lib.dllm_hip_trainer_profile(t.handle, 1))
        t.step(windows[rows], 0.0, step, weight_decay=0.0)
        seen = []
        for read in reads:
            n, ms, flops = C.c_int64(), C.c_double(), C.c_double()
            kernels.check(read(t.handle, C.byref(n), C.byref(ms), C.byref(flops)))
            assert (ms.value > 0.0 and flops.value > 0.0) == (n.value > 0)
            seen.append(n.value)
        return tuple(seen)

    lib.dllm_hip_trainer_profile.argtypes = [C.c_void_p, C.c_int]
    reads = [lib.dllm_hip_trainer_profile_read, lib.dllm_hip_trainer_profile_read_int8]
    for read in reads:
        read.argtypes = [C.c_void_p, C.POINTER(C.c_int64), C.POINTER(C.c_double), C.POINTER(C.c_double)]
    t.load(weights)
    apart = launches(2048)
    assert apart[1] == 3
    t.load(hot)
    assert launches(2048) == apart  # hands its tiles back
    t.load(weights)
    rows = 2044 if other_rows else 2048
    assert [launches(rows) for _ in range(32)] == [(apart[0] - 1, 1)] * 32  # gate and up in one launch
    assert [launches(rows) for _ in range(3)] == [apart] * 3
    t.close()
