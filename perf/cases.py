"""The work this framework is timed on: what a program that decodes with it calls, at the sizes it calls it with.

Four kinds of case, each one pass through public entry points:

  stack   one pass of a dense decoder stack through `DecodeStep`: a captured graph replayed over a filled cache. One row
          is the decode step, more rows a speculative verify pass (a tree) or a chunk of a prompt (a chain).
  matvec  one linear, called eagerly as `HipCard`'s operators are: bf16, pack12, FP8 or MXFP4, a few rows of x.
  moe     one routed layer, called eagerly: `Router` and then `Experts` or `MxExpertsLayer`.
  pack    a bf16 matrix into its 12-bit form on the GPU and widened back: what preparing a 12-bit model does.

Weights are N(0, 0.02), activations, cached keys and cached values N(0, 1), as in the repository's benchmark.
"""

from __future__ import annotations

import math
import random
from typing import Any

import torch

from btb_amd import fp8, mxfp4
from btb_amd.decode import DecodeStep, Linear, StackConfig
from btb_amd.load import MxExperts
from btb_amd.moe import Experts, MxExpertsLayer, Router
from btb_amd.native import Native
from btb_amd.pack12 import P12Weight

FP8_BLOCK = 128  # FP8 checkpoints carry one scale a 128 x 128 block


def _stack(name: str, form: str, rows: int, keys: int, **shape: int) -> dict[str, Any]:
    full = dict(layers=36, hidden=2560, q_heads=32, kv_heads=8, intermediate=9728, vocab=151936)
    full.update(shape)
    return {"name": name, "kind": "stack", "form": form, "rows": rows, "keys": keys, "tree": 0, **full}


def listed() -> list[dict[str, Any]]:
    return [
        # the smallest call: one linear of a small model, one token; latency and the host's path to the launch
        {"name": "matvec_bf16_small", "kind": "matvec", "form": "bf16", "R": 2560, "C": 2048, "M": 1},
        # a block-scaled linear of a large model at the width of a verify pass (the benchmark's FP8 matrix)
        {"name": "matvec_fp8_8rows", "kind": "matvec", "form": "fp8", "R": 18432, "C": 7168, "M": 8},
        # a gpt-oss layer (interleaved rows, biases, clamped gate) for the one token of a decode step
        {"name": "moe_oss_1row", "kind": "moe", "form": "oss", "experts": 32, "top_k": 4, "hidden": 2880,
         "intermediate": 2880, "T": 1},
        # the benchmark's bf16 layer, 128 experts of which each token picks 8, for eight tokens together
        {"name": "moe_bf16_8rows", "kind": "moe", "form": "bf16", "experts": 128, "top_k": 8, "hidden": 2048,
         "intermediate": 768, "T": 8},
        # a small model early in a conversation: many short launches
        _stack("step_small", "bf16", 1, 512, layers=28, hidden=1024, q_heads=16, intermediate=3072),
        # the benchmark's step: every weight and 4096 keys once
        _stack("step_bf16", "bf16", 1, 4096),
        # the same with every linear in the 12-bit form
        _stack("step_pack12", "pack12", 1, 4096),
        # a larger model out of an FP8 checkpoint (its head stays bf16, as such checkpoints ship it)
        _stack("step_fp8", "fp8", 1, 2000, layers=32, hidden=4096, intermediate=12288),
        # the benchmark's step late in a long document
        _stack("step_long", "bf16", 1, 32000),
        # a speculative tree of eight drafted tokens checked in one pass
        {**_stack("verify_8rows", "bf16", 8, 3001), "tree": 1},
        # a prompt read in chunks of 32 tokens
        _stack("chunk_32rows", "bf16", 32, 1536),
        # a gate/up matrix packed and checked
        {"name": "pack12_matrix", "kind": "pack", "R": 19456, "C": 2560},
    ]


def _log_int(rng: random.Random, lo: float, hi: float, step: int = 1) -> int:
    return max(step, int(math.exp(rng.uniform(math.log(lo), math.log(hi)))) // step * step)


def draw(rng: random.Random) -> dict[str, Any]:
    kind = rng.choice(["stack", "stack", "stack", "matvec", "matvec", "moe", "pack"])
    if kind == "matvec":
        form = rng.choice(["bf16", "pack12", "fp8", "mxfp4"])
        # FP8 in whole scale blocks; the others' rows in what their formats' units allow, any number of rows
        C = _log_int(rng, 512, 12288, {"bf16": 8, "pack12": 16, "fp8": FP8_BLOCK, "mxfp4": 32}[form])
        R = _log_int(rng, 512, min(65536, 2.0e8 / C), FP8_BLOCK if form == "fp8" else 1)
        return {"kind": kind, "form": form, "R": R, "C": C, "M": _log_int(rng, 1, 33)}
    if kind == "moe":
        form = rng.choice(["bf16", "mxfp4", "oss"])
        E = rng.choice([16, 32, 64, 128])
        H = _log_int(rng, 1024, 4096, 32)
        I = _log_int(rng, 512, min(4096, 1.0e9 / (E * H)), 32)
        return {"kind": kind, "form": form, "experts": E, "top_k": rng.choice([2, 4, 6, 8]), "hidden": H,
                "intermediate": I, "T": _log_int(rng, 1, 33)}
    if kind == "pack":
        C = _log_int(rng, 256, 12288, 16)
        return {"kind": kind, "R": _log_int(rng, 128, 5.0e7 / C), "C": C}
    form = rng.choice(["bf16", "bf16", "pack12", "fp8"])
    rows = rng.choice([1, 1, 1, rng.randint(2, 32)])
    hidden = _log_int(rng, 512, 4096, FP8_BLOCK if form == "fp8" else 32)
    kv_heads = rng.choice([2, 4, 8])
    q_heads = kv_heads * rng.choice([2, 4, 8] if kv_heads < 8 else [2, 4])
    inter = _log_int(rng, 2 * hidden, 4 * hidden, FP8_BLOCK if form == "fp8" else 32)
    per_layer = hidden * 128 * (2 * q_heads + 2 * kv_heads) + 3 * hidden * inter
    vocab = rng.choice([32000, 50257, 128256, 151936])
    layers = max(2, min(rng.randint(4, 36), int(3.0e9 / per_layer)))
    return {"kind": "stack", "form": form, "rows": rows, "keys": _log_int(rng, 64, 32768), "tree": int(1 < rows <= 16),
            "layers": layers, "hidden": hidden, "q_heads": q_heads, "kv_heads": kv_heads, "intermediate": inter,
            "vocab": vocab}


# ---------------------------------------------------------------------------------------------------------------------


class _Made:
    """seeded tensors on the GPU, each drawn after the one before it"""

    def __init__(self, seed: int) -> None:
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape: int, std: float = 1.0) -> torch.Tensor:
        return torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float32).mul_(std)

    def bf16(self, *shape: int, std: float = 1.0) -> torch.Tensor:
        return self.normal(*shape, std=std).to(torch.bfloat16)

    def ints(self, n: int, below: int) -> torch.Tensor:
        return torch.randint(0, below, (n,), generator=self.g, device="cuda", dtype=torch.int32)


def _config(case: dict[str, Any]) -> StackConfig:
    return StackConfig(layers=case["layers"], hidden=case["hidden"], q_heads=case["q_heads"], kv_heads=case["kv_heads"],
                       head_dim=128, intermediate=case["intermediate"], vocab=case["vocab"])


def _fp8_weight(made: _Made, rows: int, cols: int, std: float = 0.02) -> fp8.F8Weight:
    q, scales = fp8.quantize(made.normal(rows, cols, std=std), (FP8_BLOCK, FP8_BLOCK))
    return fp8.F8Weight(q, scales, rows, cols)


def _stack_weights(card: Any, cfg: StackConfig, form: str, made: _Made) -> dict[str, Any]:
    """a stack as `load_stack` hands it to `DecodeStep`: every linear in the stored form, norms and embedding bf16. Out
    of an FP8 store the head is the (tied) bf16 embedding, as such checkpoints ship it; else it is stored like the rest.
    The residual stream is of unit size and each block's output small against it, as in a trained model: embedding rows
    N(0, 1), the projections back into the stream scaled by 1 / sqrt(2 layers)."""
    H, I, D = cfg.hidden, cfg.intermediate, cfg.head_dim

    def mat(rows: int, cols: int, std: float = 0.02) -> Linear:
        if form == "fp8":
            return Linear(card, _fp8_weight(made, rows, cols, std))
        t = made.bf16(rows, cols, std=std)
        return Linear(card, P12Weight.pack(t, card) if form == "pack12" else t)

    back = 0.02 / math.sqrt(2.0 * cfg.layers)
    w: dict[str, Any] = {}
    for i in range(cfg.layers):
        p = f"layers.{i}."
        w[p + "qkv"] = mat(cfg.qkv_rows, H)
        w[p + "o"] = mat(H, cfg.q_heads * D, back)
        w[p + "gu"] = mat(2 * I, H)
        w[p + "down"] = mat(H, I, back)
        for name, n in (("ln1", H), ("ln2", H), ("wq", D), ("wk", D)):
            w[p + name] = torch.ones(n, dtype=torch.bfloat16, device="cuda")
    w["embed"] = made.bf16(cfg.vocab, H)
    w["norm"] = torch.ones(H, dtype=torch.bfloat16, device="cuda")
    w["head"] = Linear(card, w["embed"]) if form == "fp8" else mat(cfg.vocab, H)
    return w


def _prepare_stack(card: Any, case: dict[str, Any], seed: int) -> dict[str, Any]:
    cfg, T, keys = _config(case), case["rows"], case["keys"]
    made = _Made(seed)
    weights = _stack_weights(card, cfg, case["form"], made)
    # room for what the program generates next: a tenth of the context, 64 tokens at least, in whole 64s
    cap = -(-(keys + T + max(64, keys // 10)) // 64) * 64
    step = DecodeStep(card, cfg, weights, cap, T=T)
    for i in range(cfg.layers):
        step.kv[i, :, :, :keys].copy_(made.normal(2, cfg.kv_heads, keys, cfg.head_dim))
    if case["tree"]:  # every other drafted token continues the last, the ones between are second guesses
        step.set_tree([-1 if t == 0 else t - 1 if t % 2 else max(t - 2, 0) for t in range(T)])
    ids = made.ints(T, cfg.vocab)
    step.reset(keys, 0)
    step.capture(warmup=1)
    return {"kind": "stack", "step": step, "keys": keys, "ids": ids, "first": int(ids[0])}


def _prepare_matvec(card: Any, case: dict[str, Any], made: _Made) -> dict[str, Any]:
    R, C, form = case["R"], case["C"], case["form"]
    if form == "fp8":
        w, op = _fp8_weight(made, R, C), card.gemv_fp8
    elif form == "mxfp4":
        blocks, scales = mxfp4.quantize(made.normal(R, C, std=0.02))
        w, op = mxfp4.MxWeight(blocks.reshape(-1), scales.reshape(-1), R, C), card.gemv_mx4
    elif form == "pack12":
        w, op = P12Weight.pack(made.bf16(R, C, std=0.02), card), card.gemv_p12
    else:
        w, op = made.bf16(R, C, std=0.02), card.gemv
    return {"kind": "matvec", "op": op, "w": w, "x": made.bf16(case["M"], C),
            "y": torch.empty(case["M"], R, dtype=torch.bfloat16, device="cuda")}


def _prepare_moe(card: Any, case: dict[str, Any], made: _Made) -> dict[str, Any]:
    E, H, I, form = case["experts"], case["hidden"], case["intermediate"], case["form"]
    router = Router(card, made.bf16(E, H, std=0.02), case["top_k"])
    if form == "bf16":
        experts: Any = Experts(card, made.bf16(E, 2 * I, H, std=0.02), made.bf16(E, H, I, std=0.02))
    else:
        parts = []
        for rows, cols in ((2 * I, H), (H, I)):
            blocks, scales = [], []
            for _ in range(E):
                b, s = mxfp4.quantize(made.normal(rows, cols, std=0.02))
                blocks.append(b)
                scales.append(s)
            parts += [torch.stack(blocks), torch.stack(scales)]
        biases = [made.bf16(E, 2 * I, std=0.02), made.bf16(E, H, std=0.02)] if form == "oss" else [None, None]
        experts = MxExpertsLayer(card, MxExperts(*parts, *biases), oss=form == "oss")
    return {"kind": "moe", "router": router, "experts": experts, "x": made.bf16(case["T"], H)}


def prepare(case: dict[str, Any], seed: int) -> dict[str, Any]:
    card = Native.card_kernels()
    if case["kind"] == "stack":
        return _prepare_stack(card, case, seed)
    made = _Made(seed)
    if case["kind"] == "matvec":
        return _prepare_matvec(card, case, made)
    if case["kind"] == "moe":
        return _prepare_moe(card, case, made)
    return {"kind": "pack", "card": card, "t": made.bf16(case["R"], case["C"], std=0.02)}


def run(state: dict[str, Any]) -> Any:
    kind = state["kind"]
    if kind == "stack":
        step, keys = state["step"], state["keys"]
        step.reset(keys, state["first"])
        if step.T > 1:
            step.ids.copy_(state["ids"])
        step.replay()
        # every row's logits, and the K / V rows the pass has added to every layer's cache
        return {"logits": step.logits, "kv": step.kv[:, :, :, keys : keys + step.T]}
    if kind == "matvec":
        return state["op"](state["w"], state["x"], state["y"])
    if kind == "moe":
        logits, weights, picks = state["router"](state["x"])
        return {"logits": logits, "weights": weights, "picks": picks, "y": state["experts"](state["x"], picks, weights)}
    w = P12Weight.pack(state["t"], state["card"])
    R, C = w.shape
    wide = state["card"].p12_widen(w.lo, w.hi4, w.table, w.esc_idx, w.esc_val, R * C, (R, C))
    # the escape list itself is as long as the values make it; what it holds is in the rows' words and in `wide`
    return {"lo": w.lo, "hi4": w.hi4, "table": w.table, "pairs": w.pairs, "row_ptr": w.row_ptr, "row_esc": w.row_esc,
            "wide": wide}


# bytes a weight is stored in
_BYTES = {"bf16": 2.0, "pack12": 1.5, "fp8": 1.0 + 4.0 / FP8_BLOCK**2, "mxfp4": 17 / 32, "oss": 17 / 32}


def work(case: dict[str, Any]) -> dict[str, float]:
    if case["kind"] == "stack":
        cfg, T, keys, b = _config(case), case["rows"], case["keys"], _BYTES[case["form"]]
        head = cfg.vocab * cfg.hidden
        linears = cfg.weight_elements()
        per_key = 2 * cfg.kv_heads * cfg.head_dim * 2 * cfg.layers  # a K row and a V row a kv head a layer
        return {"bytes": (linears - head) * b + head * (2.0 if case["form"] == "fp8" else b)
                + (keys + T) * per_key + T * 2 * (cfg.hidden + cfg.vocab),
                "flops": 2.0 * T * linears + 4.0 * T * cfg.layers * cfg.q_heads * cfg.head_dim * (keys + T / 2)}
    if case["kind"] == "matvec":
        R, C, M = case["R"], case["C"], case["M"]
        return {"bytes": R * C * _BYTES[case["form"]] + 2 * M * (R + C), "flops": 2.0 * M * R * C}
    if case["kind"] == "moe":
        E, k, H, I, T = case["experts"], case["top_k"], case["hidden"], case["intermediate"], case["T"]
        picked = E * (1 - (1 - k / E) ** T)  # the experts that T tokens' picks name, each streamed once
        return {"bytes": picked * 3 * H * I * _BYTES[case["form"]] + 2 * E * H + 4 * T * H,
                "flops": 6.0 * T * k * H * I + 2.0 * T * E * H}
    n = float(case["R"] * case["C"])
    # 2 bytes read and 1.5 written a weight, the same back; the 8 or 16 escape words and the offset of every row
    return {"bytes": 7 * n + case["R"] * (4 + (32 if case["C"] <= 4096 else 64)), "flops": 0.0}


def tolerance(case: dict[str, Any]) -> Any:
    """Measured against torch evaluations at the same rounding points (stacks) and in 64 bits (the operators), over the
    listed cases and thirty drawn ones: a matvec rel 1.7e-3, max 3.9e-3 - its bf16 outputs' own rounding -, an expert
    layer 6e-3 / 2.4e-2, a stack of 36 layers 1.8e-2 / 8.6e-2. About four times that is stated, a stack's rel less."""
    if case["kind"] == "pack":
        return "exact"
    if case["kind"] == "matvec":
        return {"rel": 7e-3, "max": 1.6e-2}
    if case["kind"] == "moe":  # the picked experts are whole numbers and the same
        return {"rel": 2e-2, "max": 0.1, "differ": 0.0}
    return {"rel": 0.03, "max": 0.35}
