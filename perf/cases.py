"""The calls whose time is tracked: what a fine-tuning program has this library do, on data in GPU memory.

A case is a dict of plain values; its "op" names the entry point. The kernel entry points are called through the C ABI
on torch tensors, the trainer through etalii_dllm_amd.trainer. Every result is defined bit for bit (one double
accumulator per output, in a fixed order), so the tolerance of every case is "exact".

Shapes are those of the models that bench.py and the tests use: Qwen2.5-0.5B (hidden 896, intermediate 4864),
Qwen2.5-1.5B (1536, 8960, 12/2 heads of 128, vocabulary 151936), Qwen3-0.6B's attention (16/8 heads of 128),
SmolLM2-135M and OLMoE-1B-7B.
"""

from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from etalii_dllm_amd import kernels as K
from etalii_dllm_amd.trainer import Decoder, Trainer

# ---- the cases ----

SMOLLM2 = dict(vocab=49152, hidden=576, inter=1536, layers=30, heads=9, kv_heads=3, head_dim=64, theta=1e5, tied=True,
               bias=False, experts=0, topk=0, expert_inter=0)
# two of Qwen2.5-1.5B's 28 layers and two of OLMoE-1B-7B's 16: the layers repeat the same launches
QWEN25 = dict(vocab=151936, hidden=1536, inter=8960, layers=2, heads=12, kv_heads=2, head_dim=128, theta=1e6,
              tied=True, bias=True, experts=0, topk=0, expert_inter=0)
OLMOE = dict(vocab=50304, hidden=2048, inter=1024, layers=2, heads=16, kv_heads=16, head_dim=128, theta=1e4,
             tied=False, bias=False, experts=64, topk=8, expert_inter=1024)


def listed() -> list[dict]:
    return [
        # one token through a gate projection: the smallest call, launch latency and one read of the weight
        dict(name="linear_token", op="linear", rows=1, inf=896, outf=4864, bias=False),
        # a preference pair's or evaluation window's forward pass: one odd-length window
        dict(name="linear_window", op="linear", rows=1023, inf=1536, outf=8960, bias=True),
        # the backward of a short window's MLP projection with its bias gradient
        dict(name="linear_backward_window", op="linear_backward", rows=2048, inf=896, outf=4864, bias=True),
        # the backward of a whole batch's largest layer matrix (8 windows of 1024 rows)
        dict(name="linear_backward_batch", op="linear_backward", rows=8192, inf=1536, outf=8960, bias=False),
        # causal grouped-query attention over one window, forward
        dict(name="attention_window", op="attention", tokens=1024, heads=12, kv_heads=2, head_dim=128),
        # its backward over a long, odd window
        dict(name="attention_backward_long", op="attention_backward", tokens=2047, heads=16, kv_heads=8, head_dim=128),
        # a batch's norm backward with the weight's gradient (row sums and column sums)
        dict(name="rms_norm_backward_batch", op="rms_norm_backward", rows=8192, dim=1536),
        # one window's loss and logit gradient over a large vocabulary
        dict(name="cross_entropy_window", op="cross_entropy", rows=1023, vocab=151936),
        # a token through a Q8_0 projection (a quantised model read after fine-tuning)
        dict(name="linear_q8_token", op="linear_q8", rows=1, inf=1536, outf=8960),
        # whole fine-tuning steps (forward, backward, clip, AdamW): a small model at its full depth ...
        dict(name="step_smollm2", op="step", windows="256,256,256,256", aux=0.0, **SMOLLM2),
        # ... the large dense model's layers and head at batch 8 x 1024 ...
        dict(name="step_qwen2_5", op="step", windows="1024,1024,1024,1024,1024,1024,1024,1024", aux=0.0, **QWEN25),
        # ... and routed experts with the load-balancing loss on ragged windows
        dict(name="step_olmoe", op="step", windows="2048,2048,1337,500", aux=0.01, **OLMOE),
    ]


def _log_int(rng, lo: int, hi: int, multiple: int = 1) -> int:
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return min(max(v // multiple * multiple, lo), hi)


def draw(rng) -> dict:
    """A case of the same ranges: rows from one to a batch, layer sizes of small to large models, odd lengths."""
    op = rng.choice(["linear", "linear", "linear_backward", "linear_backward", "attention", "attention_backward",
                     "rms_norm_backward", "cross_entropy", "linear_q8", "step", "step"])
    # layer sizes are whole multiples of 32 in the models; every eighth draw takes any size
    m = 1 if rng.random() < 0.125 else 32
    if op in ("linear", "linear_backward"):
        return dict(op=op, rows=_log_int(rng, 1, 8192), inf=_log_int(rng, 256, 8960, m),
                    outf=_log_int(rng, 256, 8960, m), bias=rng.random() < 0.5) if m == 32 else \
            dict(op=op, rows=_log_int(rng, 1, 4096), inf=_log_int(rng, 256, 2048), outf=_log_int(rng, 256, 2048),
                 bias=rng.random() < 0.5)
    if op in ("attention", "attention_backward"):
        kv = rng.choice([1, 2, 3, 4, 8])
        return dict(op=op, tokens=_log_int(rng, 16, 2048), heads=kv * rng.choice([1, 2, 3, 4]), kv_heads=kv,
                    head_dim=rng.choice([64, 96, 128]))
    if op == "rms_norm_backward":
        return dict(op=op, rows=_log_int(rng, 1, 8192), dim=_log_int(rng, 256, 4096, m))
    if op == "cross_entropy":
        return dict(op=op, rows=_log_int(rng, 1, 2048), vocab=_log_int(rng, 1000, 151936))
    if op == "linear_q8":
        return dict(op=op, rows=_log_int(rng, 1, 2048), inf=_log_int(rng, 256, 8960, 32),
                    outf=_log_int(rng, 256, 8960, 32))
    heads = rng.choice([4, 8, 12])
    head_dim = rng.choice([64, 128])
    routed = rng.random() < 0.3
    windows = [_log_int(rng, 16, 1024) for _ in range(rng.randint(1, 8))]
    return dict(op="step", windows=",".join(map(str, windows)), aux=0.01 if routed else 0.0,
                vocab=_log_int(rng, 1024, 65536, 32), hidden=_log_int(rng, 512, 2048, 32),
                inter=_log_int(rng, 512, 6144, 32), layers=rng.randint(1, 4), heads=heads,
                kv_heads=heads // rng.choice([1, 2, 4]), head_dim=head_dim, theta=1e4, tied=rng.random() < 0.5,
                bias=rng.random() < 0.5, experts=16 if routed else 0, topk=4 if routed else 0,
                expert_inter=512 if routed else 0)


# ---- inputs ----


def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, scale: float = 1.0) -> torch.Tensor:
    return torch.randn(*shape, generator=g, device="cuda") * scale


def _activations(g, rows: int, dim: int) -> torch.Tensor:
    """Normed activations: Gaussian rows with channels of unequal size, as trained norms leave them."""
    return _randn(g, rows, dim) * torch.exp(0.5 * _randn(g, dim))


def _gradients(g, rows: int, dim: int) -> torch.Tensor:
    """Upstream gradients: small Gaussians, the rows (tokens) of unequal size."""
    return _randn(g, rows, dim, scale=1e-3) * torch.exp(0.5 * _randn(g, rows, 1))


def _workspace(nbytes: int) -> torch.Tensor:
    return torch.empty(max(int(nbytes), 1), dtype=torch.uint8, device="cuda")


def _inputs(case: dict, seed: int) -> dict:
    g, op = _gen(seed), case["op"]
    if op in ("linear", "linear_backward"):
        rows, inf, outf = case["rows"], case["inf"], case["outf"]
        s = dict(x=_activations(g, rows, inf), w=_randn(g, outf, inf, scale=0.02))
        if op == "linear":
            s["b"] = _randn(g, outf, scale=0.1) if case["bias"] else None
        else:
            s["dy"] = _gradients(g, rows, outf)
        return s
    if op in ("attention", "attention_backward"):
        t, h, kv, hd = case["tokens"], case["heads"], case["kv_heads"], case["head_dim"]
        s = dict(q=_randn(g, t, h, hd), k=_randn(g, t, kv, hd), v=_randn(g, t, kv, hd))
        if op == "attention_backward":
            s["dout"] = _gradients(g, t, h * hd).view(t, h, hd)
        return s
    if op == "rms_norm_backward":
        return dict(x=_activations(g, case["rows"], case["dim"]), w=1.0 + _randn(g, case["dim"], scale=0.1),
                    dy=_gradients(g, case["rows"], case["dim"]))
    if op == "cross_entropy":
        return dict(logits=_randn(g, case["rows"], case["vocab"], scale=2.0),
                    targets=torch.randint(0, case["vocab"], (case["rows"],), generator=g, device="cuda"))
    if op == "linear_q8":
        return dict(x=_activations(g, case["rows"], case["inf"]),
                    w=_randn(g, case["outf"], case["inf"], scale=0.02))
    raise ValueError(op)


# ---- the model of the step cases ----


def _lengths(case: dict) -> list[int]:
    return [int(n) for n in case["windows"].split(",")]


def _shapes(case: dict) -> dict[str, tuple[int, ...]]:
    H, q, kv = case["hidden"], case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
    shapes = {"token_embedding.weight": (case["vocab"], H), "final_norm.weight": (H,)}
    if not case["tied"]:
        shapes["lm_head.weight"] = (case["vocab"], H)
    for i in range(case["layers"]):
        p = f"layers.{i}."
        shapes.update({p + "attention_norm.weight": (H,), p + "mlp_norm.weight": (H,),
                       p + "attention.q.weight": (q, H), p + "attention.k.weight": (kv, H),
                       p + "attention.v.weight": (kv, H), p + "attention.o.weight": (H, q)})
        if case["bias"]:
            shapes.update({p + "attention.q.bias": (q,), p + "attention.k.bias": (kv,),
                           p + "attention.v.bias": (kv,)})
        if case["experts"]:
            shapes[p + "mlp.router.weight"] = (case["experts"], H)
            blocks = [(f"{p}mlp.experts.{e}.", case["expert_inter"]) for e in range(case["experts"])]
        else:
            blocks = [(p + "mlp.", case["inter"])]
        for x, ei in blocks:
            shapes.update({x + "gate.weight": (ei, H), x + "up.weight": (ei, H), x + "down.weight": (H, ei)})
    return shapes


def _weights(case: dict, seed: int):
    """(name, tensor) of every weight: N(0, 0.02) matrices and biases, norms near one."""
    g = _gen(seed)
    for name, shape in _shapes(case).items():
        if name.endswith("norm.weight"):
            yield name, 1.0 + _randn(g, *shape, scale=0.1)
        else:
            yield name, _randn(g, *shape, scale=0.02)


def _token_windows(case: dict, seed: int) -> list[list[int]]:
    rng = np.random.default_rng(seed)
    return [rng.integers(0, case["vocab"], n + 1).tolist() for n in _lengths(case)]


class _View:
    """Device memory of a trainer as something torch.as_tensor reads without a copy. The tensor keeps this object, and
    with it the trainer that owns the memory, alive."""

    def __init__(self, trainer: Trainer, ptr: int, numel: int) -> None:
        self.trainer = trainer
        self.__cuda_array_interface__ = dict(shape=(numel,), typestr="<f4", data=(ptr, False), version=2)


def _layout(case: dict) -> tuple[dict[str, int], int]:
    """Where each tensor lies in the trainer's parameter memory: natural order, each 256-byte aligned (64 floats)."""
    offsets, end = {}, 0
    shapes = _shapes(case)
    for name in sorted(shapes, key=_natural):
        offsets[name] = end
        end += -(-math.prod(shapes[name]) // 64) * 64
    return offsets, end


def _parameters(trainer: Trainer, case: dict) -> torch.Tensor:
    """All parameters as one flat view (a program that hands them on wants one buffer, not hundreds)."""
    offsets, end = _layout(case)
    base = None
    for name, shape in _shapes(case).items():
        ptr, numel = C.c_void_p(), C.c_int64()
        K.check(K.lib.dllm_hip_trainer_tensor(trainer.handle, name.encode(), Trainer.PARAM, C.byref(ptr),
                                              C.byref(numel)))
        at = ptr.value - 4 * offsets[name]
        base = at if base is None else base
        assert numel.value == math.prod(shape) and at == base, name
    return torch.as_tensor(_View(trainer, base, end), device="cuda")


ADAMW = dict(learning_rate=1e-4, beta1=0.9, beta2=0.999, eps=1e-8, weight_decay=0.01, max_grad_norm=1.0)


def _prepare_step(case: dict, seed: int) -> dict:
    lengths = _lengths(case)
    decoder = Decoder(case["vocab"], case["hidden"], case["inter"], case["layers"], case["heads"], case["kv_heads"],
                      case["head_dim"], 1e-6, case["theta"], case["tied"], attention_bias=case["bias"],
                      experts=case["experts"], experts_per_token=case["topk"],
                      expert_intermediate=case["expert_inter"])
    trainer = Trainer(decoder, sum(lengths), len(lengths), max(lengths))
    params, (offsets, _) = _parameters(trainer, case), _layout(case)
    params.zero_()
    for name, values in _weights(case, seed):
        params[offsets[name]:offsets[name] + values.numel()].copy_(values.view(-1))
    torch.cuda.synchronize()
    return dict(op="step", trainer=trainer, params=params, windows=_token_windows(case, seed), aux=case["aux"], step=0)


def prepare(case: dict, seed: int) -> dict:
    op = case["op"]
    if op == "step":
        return _prepare_step(case, seed)
    s = _inputs(case, seed)
    s.update(op=op, case=case)
    lib = K.lib
    if op == "linear":
        s["out"] = torch.empty(case["rows"], case["outf"], device="cuda")
        s["ws"] = _workspace(lib.dllm_hip_linear_workspace(case["rows"], case["inf"], case["outf"]))
    elif op == "linear_backward":
        s["dx"], s["dw"] = torch.empty_like(s["x"]), torch.empty_like(s["w"])
        s["db"] = torch.empty(case["outf"], device="cuda") if case["bias"] else None
        s["ws"] = _workspace(lib.dllm_hip_linear_backward_workspace(case["rows"], case["inf"], case["outf"]))
    elif op in ("attention", "attention_backward"):
        t, h, kv, hd = case["tokens"], case["heads"], case["kv_heads"], case["head_dim"]
        query = getattr(lib, f"dllm_hip_{op}_workspace")
        s["ws"] = _workspace(query(t, t, h, kv, hd, hd, 1, 0, 0, 0.0))
        if op == "attention":
            s["out"] = torch.empty_like(s["q"])
        else:
            s["dq"], s["dk"], s["dv"] = (torch.empty_like(s[n]) for n in "qkv")
    elif op == "rms_norm_backward":
        s["dx"], s["dw"] = torch.empty_like(s["x"]), torch.empty_like(s["w"])
        s["ws"] = _workspace(lib.dllm_hip_rms_norm_backward_workspace(case["rows"]))
    elif op == "cross_entropy":
        s["dlogits"] = torch.empty_like(s["logits"])
        s["ws"] = _workspace(lib.dllm_hip_cross_entropy_workspace(case["rows"]))
    elif op == "linear_q8":
        w = s.pop("w")
        s["wq"] = torch.empty(w.shape, dtype=torch.int8, device="cuda")
        s["ws_scales"] = torch.empty(w.shape[0], w.shape[1] // 32, device="cuda")
        K.check(lib.dllm_hip_quantize_q8_0(w.data_ptr(), s["wq"].data_ptr(), s["ws_scales"].data_ptr(), w.numel(),
                                           _stream()))
        torch.cuda.synchronize()  # w is freed here
        s["out"] = torch.empty(case["rows"], case["outf"], device="cuda")
        s["ws"] = _workspace(lib.dllm_hip_linear_q8_workspace(case["rows"], case["inf"]))
    return s


# ---- one pass ----


def _stream() -> int:
    return torch.cuda.current_stream().cuda_stream


def _ptr(t):
    return None if t is None else t.data_ptr()


def run(state: dict):
    s, lib, op = state, K.lib, state["op"]
    if op == "step":
        s["step"] += 1
        loss, norm = s["trainer"].step(s["windows"], ADAMW["learning_rate"], s["step"], router_aux_loss=s["aux"])
        return {"loss": loss, "norm": norm, "params": s["params"]}
    c, ws = s["case"], s["ws"]
    if op == "linear":
        K.check(lib.dllm_hip_linear(s["x"].data_ptr(), s["w"].data_ptr(), _ptr(s["b"]), s["out"].data_ptr(),
                                    c["rows"], c["inf"], c["outf"], ws.data_ptr(), ws.numel(), _stream()))
        return s["out"]
    if op == "linear_backward":
        K.check(lib.dllm_hip_linear_backward(s["x"].data_ptr(), s["w"].data_ptr(), s["dy"].data_ptr(),
                                             s["dx"].data_ptr(), s["dw"].data_ptr(), _ptr(s["db"]), c["rows"],
                                             c["inf"], c["outf"], ws.data_ptr(), ws.numel(), _stream()))
        return [s["dx"], s["dw"]] + ([s["db"]] if s["db"] is not None else [])
    if op in ("attention", "attention_backward"):
        t, h, kv, hd = c["tokens"], c["heads"], c["kv_heads"], c["head_dim"]
        shape = (t, t, h, kv, hd, hd, 1.0 / math.sqrt(hd), 1, 0, 0, 0.0, ws.data_ptr(), ws.numel(), _stream())
        ins = [s[n].data_ptr() for n in "qkv"]
        if op == "attention":
            K.check(lib.dllm_hip_attention(*ins, s["out"].data_ptr(), *shape))
            return s["out"]
        K.check(lib.dllm_hip_attention_backward(*ins, s["dout"].data_ptr(), s["dq"].data_ptr(), s["dk"].data_ptr(),
                                                s["dv"].data_ptr(), *shape))
        return [s["dq"], s["dk"], s["dv"]]
    if op == "rms_norm_backward":
        K.check(lib.dllm_hip_rms_norm_backward(s["x"].data_ptr(), s["w"].data_ptr(), s["dy"].data_ptr(),
                                               s["dx"].data_ptr(), s["dw"].data_ptr(), c["rows"], c["dim"], 1e-6, 0,
                                               ws.data_ptr(), ws.numel(), _stream()))
        return [s["dx"], s["dw"]]
    if op == "cross_entropy":
        loss = C.c_double()
        K.check(lib.dllm_hip_cross_entropy(s["logits"].data_ptr(), s["targets"].data_ptr(), s["dlogits"].data_ptr(),
                                           c["rows"], c["vocab"], 1.0 / c["rows"], C.byref(loss), ws.data_ptr(),
                                           ws.numel(), _stream()))
        return [s["dlogits"], loss.value]
    if op == "linear_q8":
        K.check(lib.dllm_hip_linear_q8(s["x"].data_ptr(), s["wq"].data_ptr(), s["ws_scales"].data_ptr(), None,
                                       s["out"].data_ptr(), c["rows"], c["inf"], c["outf"], ws.data_ptr(),
                                       ws.numel(), _stream()))
        return s["out"]
    raise ValueError(op)


# ---- what a pass cannot do without ----


def work(case: dict) -> dict:
    op = case["op"]
    if op in ("linear", "linear_backward"):
        r, i, o = case["rows"], case["inf"], case["outf"]
        if op == "linear":
            return {"bytes": 4.0 * (r * i + i * o + r * o), "flops": 2.0 * r * i * o}
        return {"bytes": 4.0 * (2 * r * i + 2 * i * o + r * o), "flops": 4.0 * r * i * o}
    if op in ("attention", "attention_backward"):
        t, h, kv, hd = case["tokens"], case["heads"], case["kv_heads"], case["head_dim"]
        pairs = h * t * (t + 1) / 2
        if op == "attention":
            return {"bytes": 4.0 * t * hd * (2 * h + 2 * kv), "flops": 4.0 * hd * pairs}
        return {"bytes": 4.0 * t * hd * (3 * h + 4 * kv), "flops": 10.0 * hd * pairs}
    if op == "rms_norm_backward":
        return {"bytes": 12.0 * case["rows"] * case["dim"], "flops": 12.0 * case["rows"] * case["dim"]}
    if op == "cross_entropy":
        return {"bytes": 8.0 * case["rows"] * case["vocab"], "flops": 6.0 * case["rows"] * case["vocab"]}
    if op == "linear_q8":
        r, i, o = case["rows"], case["inf"], case["outf"]
        return {"bytes": 4.0 * r * (i + o) + o * i * (1.0 + 4.0 / 32), "flops": 2.0 * r * i * o}
    lengths = _lengths(case)
    tokens = sum(lengths)
    H, q, kv = case["hidden"], case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
    if case["experts"]:
        mlp = case["experts"] * H + case["topk"] * 3 * H * case["expert_inter"]
    else:
        mlp = 3 * H * case["inter"]
    matmul = case["layers"] * (2 * H * q + 2 * H * kv + mlp) + case["vocab"] * H
    pairs = sum(n * (n + 1) / 2 for n in lengths) * case["heads"] * case["layers"]
    params = sum(math.prod(s) for s in _shapes(case).values())
    # weights and both moments read and written once
    return {"bytes": 24.0 * params + 8.0 * tokens, "flops": 6.0 * matmul * tokens + 14.0 * case["head_dim"] * pairs}


def tolerance(case: dict):
    return "exact"


# ---- the same in 64 bits ----


def _attention64(q, k, v, scale):
    t, h, kv = q.shape[0], q.shape[1], k.shape[1]
    out = []
    mask = torch.ones(t, t, dtype=torch.bool, device=q.device).tril()
    for head in range(h):
        s = (q[:, head] @ k[:, head // (h // kv)].T) * scale
        p = torch.softmax(s.masked_fill(~mask, -math.inf), dim=-1)
        out.append(p @ v[:, head // (h // kv)])
    return torch.stack(out, dim=1)


def _rms64(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rope64(x, theta):
    t, _, hd = x.shape
    inv = theta ** (-torch.arange(0, hd, 2, dtype=torch.float64, device=x.device) / hd)
    ang = torch.arange(t, dtype=torch.float64, device=x.device)[:, None] * inv
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x[..., : hd // 2], x[..., hd // 2:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)


def _exact_step(case: dict, seed: int) -> dict:
    p = {n: w.double().requires_grad_() for n, w in _weights(case, seed)}
    windows = _token_windows(case, seed)
    scale = 1.0 / sum(_lengths(case))
    total = 0.0
    for win in windows:  # one window at a time bounds the logits' memory
        ids = torch.tensor(win, device="cuda")
        x = p["token_embedding.weight"][ids[:-1]]
        t = x.shape[0]
        for i in range(case["layers"]):
            a, m = f"layers.{i}.attention", f"layers.{i}.mlp"
            h = _rms64(x, p[f"{a}_norm.weight"], 1e-6)
            q, k, v = (torch.nn.functional.linear(h, p[f"{a}.{n}.weight"], p.get(f"{a}.{n}.bias")) for n in "qkv")
            q, k, v = (y.view(t, -1, case["head_dim"]) for y in (q, k, v))
            q, k = _rope64(q, case["theta"]), _rope64(k, case["theta"])
            o = _attention64(q, k, v, 1.0 / math.sqrt(case["head_dim"])).reshape(t, -1)
            x = x + o @ p[f"{a}.o.weight"].T
            h = _rms64(x, p[f"{m}_norm.weight"], 1e-6)
            gate = torch.nn.functional.silu(h @ p[f"{m}.gate.weight"].T) * (h @ p[f"{m}.up.weight"].T)
            x = x + gate @ p[f"{m}.down.weight"].T
        x = _rms64(x, p["final_norm.weight"], 1e-6)
        head = p["token_embedding.weight" if case["tied"] else "lm_head.weight"]
        loss = torch.nn.functional.cross_entropy(x @ head.T, ids[1:], reduction="sum")
        (loss * scale).backward()
        total += loss.item()
    norm = math.sqrt(sum((w.grad ** 2).sum().item() for w in p.values()))
    clip = min(1.0, ADAMW["max_grad_norm"] / norm)
    offsets, end = _layout(case)
    params = torch.zeros(end, dtype=torch.float64, device="cuda")
    with torch.no_grad():
        for name in sorted(p, key=_natural):
            w = p.pop(name)
            g = w.grad * clip
            m, v = (1 - ADAMW["beta1"]) * g, (1 - ADAMW["beta2"]) * g * g
            update = (m / (1 - ADAMW["beta1"])) / ((v / (1 - ADAMW["beta2"])).sqrt() + ADAMW["eps"])
            w = w - ADAMW["learning_rate"] * (update + ADAMW["weight_decay"] * w)
            params[offsets[name]:offsets[name] + w.numel()] = w.view(-1)
    return {"loss": total * scale, "norm": norm, "params": params}


def _natural(name: str):
    """Natural order: the numbers in a name compare as numbers, before letters."""
    import re

    return (*((0, int(p), "") if p.isdigit() else (1, 0, p) for p in re.split(r"(\d+)", name)), name)


def exact(case: dict, seed: int):
    op = case["op"]
    if op == "step":
        # the choice of experts is discrete: rounding decides near-ties, so a routed step has no 64-bit value
        return None if case["experts"] else _exact_step(case, seed)
    if op == "linear_q8":
        # the path is defined on the quantised blocks: float32 scales and int8 values, exact in 64 bits
        s = prepare(case, seed)
        x = s["x"].view(case["rows"], -1, 32)
        scale = (x.abs().amax(-1, keepdim=True) / 127.0).float()
        inv = torch.where(scale > 0, 1.0 / scale, torch.zeros_like(scale))
        xq = torch.round(x * inv).clamp(-127, 127).double() * scale.double()
        w = s["wq"].view(case["outf"], -1, 32).double() * s["ws_scales"].double()[..., None]
        return xq.view(case["rows"], -1) @ w.view(case["outf"], -1).T
    s = {k: (v.double() if v is not None and v.is_floating_point() else v) for k, v in _inputs(case, seed).items()}
    if op == "linear":
        return torch.nn.functional.linear(s["x"], s["w"], s["b"])
    if op == "linear_backward":
        return [s["dy"] @ s["w"], s["dy"].T @ s["x"]] + ([s["dy"].sum(0)] if case["bias"] else [])
    if op == "attention":
        return _attention64(s["q"], s["k"], s["v"], 1.0 / math.sqrt(case["head_dim"]))
    if op == "attention_backward":
        qkv = [s[n].requires_grad_() for n in "qkv"]
        _attention64(*qkv, 1.0 / math.sqrt(case["head_dim"])).backward(s["dout"])
        return [t.grad for t in qkv]
    if op == "rms_norm_backward":
        x, w = s["x"].requires_grad_(), s["w"].requires_grad_()
        _rms64(x, w, 1e-6).backward(s["dy"])
        return [x.grad, w.grad]
    if op == "cross_entropy":
        x = s["logits"].requires_grad_()
        loss = torch.nn.functional.cross_entropy(x, s["targets"], reduction="sum")
        (loss / case["rows"]).backward()
        return [x.grad, loss.item()]
    raise ValueError(op)
