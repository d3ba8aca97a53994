"""Decode steps over caches whose attention walks spans on the matrix cores (`attn_decode_qkv_span`): one row from 8192 slots
on, passes of more rows over spans of several batches; the same steps with a launch per operator, on the vector kernels'
spans, are the reference."""

from __future__ import annotations

import pytest
import torch

from btb_amd.decode import DecodeStep, Linear, StackConfig

from .helpers import gen

pytestmark = pytest.mark.gpu

# eight query heads a kv head and few kv heads: one row walks spans from 8192 slots on, 2 .. 32 rows over any spans
CFG = StackConfig(layers=2, hidden=256, q_heads=16, kv_heads=2, head_dim=128, intermediate=512, vocab=1000)
TOKENS = [17, 5, 901, 33, 4, 250, 7, 12]


def weights(card, off: int = 0):
    """random weights; the norms' as views `off` values into a larger tensor"""
    g = gen(1700)

    def mat(rows, cols):
        return Linear(card, (torch.randn(rows, cols, generator=g) * 0.05).to(torch.bfloat16).cuda())

    def vec(n):
        t = torch.zeros(n + 8, dtype=torch.bfloat16)
        t[off : off + n] = (1.0 + 0.1 * torch.randn(n, generator=g)).to(torch.bfloat16)
        return t.cuda()[off : off + n]

    H, I = CFG.hidden, CFG.intermediate
    w = {}
    for i in range(CFG.layers):
        p = f"layers.{i}."
        w[p + "qkv"], w[p + "o"] = mat(CFG.qkv_rows, H), mat(H, CFG.q_heads * CFG.head_dim)
        w[p + "gu"], w[p + "down"] = mat(2 * I, H), mat(H, I)
        for name, n in (("ln1", H), ("ln2", H), ("wq", CFG.head_dim), ("wk", CFG.head_dim)):
            w[p + name] = vec(n)
    w["embed"] = torch.randn(CFG.vocab, H, generator=g).to(torch.bfloat16).cuda()
    w["norm"], w["head"] = vec(H), mat(CFG.vocab, H)
    return w


def make(card, w, cap, T, n0, kv, tree=None, **kw):
    step = DecodeStep(card, CFG, w, cap, T=T, **kw)
    fill(step, n0, kv)
    if tree is not None:
        step.set_tree(tree)
    return step


def fill(step, n0, kv):
    step.kv.zero_()
    step.kv[:, :, :, :n0].copy_(kv[:, :, :, :n0])
    step.reset(n0, TOKENS[0])
    if step.T > 1:
        step.ids.copy_(torch.tensor([TOKENS[t % 8] + t for t in range(step.T)], dtype=torch.int32))


def cache(cap):
    return torch.randn(CFG.layers, 2, CFG.kv_heads, cap, CFG.head_dim, generator=torch.Generator(device="cuda").manual_seed(5),
                       device="cuda").to(torch.bfloat16)


def close(a, b):
    """logits to the step's bar (tests/test_decode_gpu.py)"""
    return float((a.float() - b.float()).abs().max()) <= 3e-2 * float(b.float().abs().max())


def follow(step, n0, kv, steps, graph):
    """logits and cache of `steps` steps, eager or replayed, with unrelated work and a synchronise between them"""
    fill(step, n0, kv)
    out = []
    for _ in range(steps):
        step.replay() if graph else step.body()
        torch.cuda.synchronize()
        out.append(step.logits.clone())
        assert bool(torch.isfinite(torch.randn(1 << 14, device="cuda").sum()))
        torch.cuda.synchronize()
    return torch.stack(out), step.kv.clone()


# the cache all but empty, one key short of a batch a span and at it (64 spans of 128), and near its end: the spans follow
# the keys from step to step
@pytest.mark.parametrize("n0", [0, 8189, 16380])
def test_one_row_on_a_long_cache(card, n0):
    """eager steps, replayed steps - the same bits - and the sequence with a launch per operator, to the step's bar; every
    one writes its row into the cache"""
    cap = 16384
    w, kv = weights(card), cache(cap)
    step, plain = DecodeStep(card, CFG, w, cap), DecodeStep(card, CFG, w, cap, fused=False)
    assert step.span_fused and step.fused and not plain.span_fused and not plain.fused
    eager, kv_e = follow(step, n0, kv, 4, False)
    fill(step, n0, kv)
    step.capture(warmup=1)
    for _ in range(2):
        again, kv_g = follow(step, n0, kv, 4, True)
        assert torch.equal(again, eager) and torch.equal(kv_g, kv_e)
    # the other sequence on the same tokens: its own picks may differ where two logits are close
    fill(step, n0, kv)
    fill(plain, n0, kv)
    for t in range(4):
        for s in (step, plain):
            s.ids.fill_(TOKENS[t])
            s.body()
        torch.cuda.synchronize()
        assert close(step.logits, plain.logits), t
    new = slice(n0, n0 + 4)
    a, b = step.kv[:, :, :, new].float(), plain.kv[:, :, :, new].float()
    assert float((a - b).abs().max()) <= 3e-2 * float(b.abs().max())
    assert torch.equal(step.kv[:, :, :, :n0], kv[:, :, :, :n0]) and not bool(step.kv[:, :, :, n0 + 4 :].any())


@pytest.mark.parametrize("T,cap", [(2, 9000), (2, 17000), (3, 17000), (20, 9000), (32, 9000)])
@pytest.mark.parametrize("tree", [False, True])
def test_passes_over_long_spans(card, T, cap, tree):
    """a pass whose attention walks spans of several batches from the fused rows, the pass's rows in the middle of the cache,
    across two spans and at its end"""
    w, kv = weights(card), cache(cap)
    par = [-1] + [t - 2 if t % 3 == 2 else t - 1 for t in range(1, T)] if tree else None
    step, plain = DecodeStep(card, CFG, w, cap, T=T), DecodeStep(card, CFG, w, cap, T=T, fused=False)
    span = -(-(-(-cap // step.S)) // 128) * 128
    assert step.span_fused and not plain.span_fused and span > 128
    for s in (step, plain):
        s.set_tree(par)
    fill(step, 5, kv)
    step.capture(warmup=1)
    for n0 in (5, 3 * span - 1, cap - T):
        fill(step, n0, kv)
        step.body()
        torch.cuda.synchronize()
        eager, kv_e = step.logits.clone(), step.kv.clone()
        fill(step, n0, kv)
        step.replay()
        fill(plain, n0, kv)
        plain.body()
        torch.cuda.synchronize()
        assert torch.equal(step.logits, eager) and torch.equal(step.kv, kv_e)
        assert close(step.logits, plain.logits), n0
        assert torch.equal(step.kv[:, :, :, :n0], kv[:, :, :, :n0]) and not bool(step.kv[:, :, :, n0 + T :].any())


def test_norm_weights_at_any_place(card):
    """norm weights that are views into a larger tensor, not 16-byte aligned: such a step keeps the kernels that take
    them, on a long cache too"""
    cap, n0 = 16384, 9000
    kv = cache(cap)
    odd, even = make(card, weights(card, 1), cap, 1, n0, kv), make(card, weights(card), cap, 1, n0, kv)
    assert even.span_fused and not odd.span_fused
    for s in (odd, even):
        s.body()
    torch.cuda.synchronize()
    assert close(odd.logits, even.logits)
    odd, even = make(card, weights(card, 1), cap, 20, n0, kv), make(card, weights(card), cap, 20, n0, kv)
    assert even.span_fused and not odd.span_fused
    for s in (odd, even):
        s.body()
    torch.cuda.synchronize()
    assert close(odd.logits, even.logits)


def test_the_knob_switches_the_walk_off(card):
    w = weights(card)
    card.set_tuning("attn_mfma", 0)
    try:
        assert not DecodeStep(card, CFG, w, 16384).span_fused and not DecodeStep(card, CFG, w, 16384, T=20).span_fused
    finally:
        card.set_tuning("attn_mfma", -1)
    assert DecodeStep(card, CFG, w, 16384).span_fused and DecodeStep(card, CFG, w, 16384, T=20).span_fused


def test_fp8_rows_the_folded_norm_has_no_room_for(card):
    """a residual stream whose two rows fit LDS but not with the norm's weight beside them: one launch per operator"""
    from btb_amd import fp8

    H, D = 32768, 128
    cfg = StackConfig(layers=1, hidden=H, q_heads=2, kv_heads=1, head_dim=D, intermediate=256, vocab=64)
    g = gen(1750)

    def f8(rows, cols):
        q, s = fp8.quantize(torch.randn(rows, cols, generator=g) * 0.01, (128, 128))
        return Linear(card, fp8.F8Weight(q.view(torch.uint8).cuda(), s.cuda(), rows, cols))

    ones = lambda n: torch.ones(n, dtype=torch.bfloat16, device="cuda")
    p = "layers.0."
    w = {p + "qkv": f8(4 * D, H), p + "o": f8(H, 2 * D), p + "gu": f8(512, H), p + "down": f8(H, 256), p + "ln1": ones(H),
         p + "ln2": ones(H), p + "wq": ones(D), p + "wk": ones(D), "norm": ones(H),
         "embed": torch.randn(64, H, generator=g).to(torch.bfloat16).cuda()}
    w["head"] = Linear(card, w["embed"])
    logits = []
    for fused in (None, False):
        step = DecodeStep(card, cfg, w, 64, T=2, fused=fused)
        assert not step.fused
        step.reset(3, 5)
        step.body()
        torch.cuda.synchronize()
        logits.append(step.logits.clone())
    assert bool(torch.isfinite(logits[0].float()).all()) and close(logits[0], logits[1])
