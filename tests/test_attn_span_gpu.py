"""The matrix-core attention that walks a span in batches of 128 keys (attn_span.hip), against f64 attention over the
keys each row sees."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import decode as od
from .helpers import gen

pytestmark = pytest.mark.gpu


def seen_by(t, n0, par, win):
    """the slots row t attends to: the cache and, of the pass's own rows, itself and its ancestors, under the window"""
    if par is None:
        slots = list(range(n0 + t + 1))
        pos = slots
    else:
        path, p = [], t
        while p >= 0:
            path.append(p)
            p = par[p]
        path = path[::-1]
        slots = list(range(n0)) + [n0 + p for p in path]
        pos = list(range(n0)) + [n0 + d for d in range(len(path))]
    return [s for s, ps in zip(slots, pos) if win == 0 or ps >= pos[-1] + 1 - win]


# one, two and four tiles of pairs a workgroup, several workgroups a kv head; the rows' own slots in the first, a middle
# and the last batch and across a batch's edge; spans with nothing to see; every group size; a row map
@pytest.mark.parametrize("n0,T,Hq,Hk,S,tree,win,mapped", [
    (1000, 2, 8, 8, 2, False, 0, False), (1000, 2, 16, 2, 3, True, 0, False), (383, 5, 8, 2, 2, False, 0, True),
    (250, 17, 32, 8, 1, False, 0, False), (0, 32, 16, 2, 1, True, 0, False), (127, 33, 8, 8, 1, False, 0, False),
    (640, 32, 8, 1, 2, False, 100, False), (500, 21, 4, 1, 2, True, 300, True), (256, 9, 16, 2, 7, False, 0, False),
    (1, 3, 8, 1, 1, True, 2, False), (2047, 8, 32, 8, 5, True, 0, False)])
def test_attention_over_long_spans(card, n0, T, Hq, Hk, S, tree, win, mapped):
    D = 128
    cap = n0 + T + 300
    g = gen(1200 + n0 + T)
    K = torch.randn(Hk, cap, D, generator=g).to(torch.bfloat16)
    V = torch.randn(Hk, cap, D, generator=g).to(torch.bfloat16)
    K[:, n0 + T:] = float("nan")  # what lies past the pass must not leak through weight 0
    V[:, n0 + T:] = float("nan")
    q = (2 * torch.randn(T, Hq * D, generator=g)).to(torch.bfloat16)
    par = [-1] + [int(torch.randint(-1, t, (1,), generator=g)) for t in range(1, T)] if tree else None
    part = None if par is None else torch.tensor(par, dtype=torch.int32, device="cuda")
    scale = 1.0 / np.sqrt(D)
    n0t = torch.tensor([n0], dtype=torch.int32, device="cuda")
    scratch = card.attn_scratch(T, Hq, Hk, D, S)
    tbl, Kd, Vd = None, K, V
    if mapped:
        order = torch.randperm(cap, generator=g)
        Kd, Vd = torch.empty_like(K), torch.empty_like(V)
        Kd[:, order], Vd[:, order] = K, V
        tbl = order.to(torch.int32).cuda()

    def run():
        att = torch.zeros(T, Hq * D, dtype=torch.bfloat16, device="cuda")
        card.attn_decode(q.cuda(), Kd.cuda(), Vd.cuda(), att, n0t, Hq, Hk, D, scale, S, scratch, par=part, win=win,
                         tbl=tbl)
        return att

    y = run()
    assert torch.equal(run(), y)
    got = y.float().cpu().numpy()
    for t in range(T):
        keep = seen_by(t, n0, par, win)
        want = od.attention(q[t].float().numpy().reshape(Hq, D), K[:, keep].float().numpy(), V[:, keep].float().numpy(),
                            scale)
        # weights and outputs are rounded to bf16 (2^-9 each), as in the other attention kernels' tests
        worst = np.abs(got[t].reshape(Hq, D) - want).max() / np.abs(want).max()
        assert worst <= 2.0**-7, (t, worst)


# one row and several; one, two and four tiles of pairs, several workgroups a kv head; the rows' own slots within one
# batch, across two and across two spans, the first and the last slot of the cache; with and without norm weights
@pytest.mark.parametrize("n0,T,Hq,Hk,S,tree", [
    (1000, 1, 16, 2, 2, False), (255, 1, 32, 8, 1, False), (256, 1, 8, 8, 2, False), (0, 1, 4, 2, 1, False),
    (1000, 2, 16, 2, 3, True), (383, 5, 8, 2, 2, False), (250, 17, 32, 8, 1, False), (0, 32, 16, 2, 1, True),
    (500, 32, 8, 8, 2, False), (250, 21, 4, 1, 2, True), (2047, 8, 32, 8, 5, True), (246, 10, 8, 1, 1, False)])
@pytest.mark.parametrize("with_norm", [True, False])
def test_long_spans_from_the_fused_qkv_rows(card, n0, T, Hq, Hk, S, tree, with_norm):
    """`attn_decode_qkv_span` against `norm_rope_kv` and `attn_decode` at the same span count: the same cache, nothing else
    in it touched, and from two rows on the same output bits (one row: both within bf16's bar of f64 attention)"""
    from btb_amd.decode import StackConfig, rope_tables

    D = 128
    cap = n0 + T
    cap = 256 if n0 + T == 256 else cap + 150
    g = gen(1300 + n0 + T)
    K = torch.randn(Hk, cap, D, generator=g).to(torch.bfloat16)
    V = torch.randn(Hk, cap, D, generator=g).to(torch.bfloat16)
    K[:, n0:] = float("nan")
    V[:, n0:] = float("nan")
    qkv = torch.randn(T, (Hq + 2 * Hk) * D, generator=g).to(torch.bfloat16).cuda()
    wn = (1 + 0.1 * torch.randn(D, generator=g)).to(torch.bfloat16).cuda() if with_norm else None
    cos, sin = rope_tables(StackConfig(q_heads=Hq, kv_heads=Hk), cap + 64, torch.device("cuda"))
    par = [-1] + [int(torch.randint(-1, t, (1,), generator=g)) for t in range(1, T)] if tree else None
    part, depth = None, None
    if tree:
        d = []
        for p in par:
            d.append(0 if p < 0 else d[p] + 1)
        part = torch.tensor(par, dtype=torch.int32, device="cuda")
        depth = torch.tensor(d, dtype=torch.int32, device="cuda")
    scale = 1.0 / np.sqrt(D)
    n0t = torch.tensor([n0], dtype=torch.int32, device="cuda")
    scratch = card.attn_scratch(T, Hq, Hk, D, S)
    K1, V1, K2, V2 = K.cuda(), V.cuda(), K.cuda(), V.cuda()
    q = torch.empty(T, Hq * D, dtype=torch.bfloat16, device="cuda")
    want, got = torch.zeros_like(q), torch.zeros_like(q)
    card.norm_rope_kv(qkv, wn, wn, 1e-6, cos, sin, n0t, K1, V1, q, Hq, Hk, D, depth=depth)
    card.attn_decode(q, K1, V1, want, n0t, Hq, Hk, D, scale, S, scratch, par=part)
    card.attn_decode_qkv_span(qkv, wn, wn, 1e-6, cos, sin, n0t, K2, V2, got, Hq, Hk, D, scale, S, scratch, depth=depth,
                              par=part)
    for a, b in ((K1, K2), (V1, V2)):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    span = -(-(-(-cap // S)) // 128) * 128
    if T > 1 and not (span == 128 and Hq // Hk in (2, 4)):  # there attn_decode is the one-batch kernel
        assert torch.equal(want.view(torch.int16), got.view(torch.int16))
    assert bool(torch.isfinite(got.float()).all())
    for t in range(T):
        keep = seen_by(t, n0, par, 0)
        ref = od.attention(q[t].float().cpu().numpy().reshape(Hq, D), K1[:, keep].float().cpu().numpy(),
                           V1[:, keep].float().cpu().numpy(), scale)
        worst = np.abs(got[t].float().cpu().numpy().reshape(Hq, D) - ref).max() / np.abs(ref).max()
        assert worst <= 2.0**-7, (t, worst)


# one row and several, from the fused rows and from q; one, two and four tiles of pairs; passes of more than sixteen rows
# over spans of one batch (the one-batch kernel's two terms); few keys, whose weights are heaviest, and many
@pytest.mark.parametrize("n0,T,Hq,Hk,S", [(9000, 1, 32, 8, 16), (20000, 1, 8, 2, 32), (100, 2, 32, 4, 1), (1500, 3, 16, 2, 4),
                                          (6000, 8, 32, 8, 16), (700, 12, 8, 8, 3), (1536, 32, 32, 8, 13),
                                          (300, 17, 16, 8, 3), (260, 32, 8, 2, 3), (3000, 26, 32, 8, 6), (5000, 32, 16, 2, 8)])
def test_weights_lose_nothing_the_output_would_show(card, n0, T, Hq, Hk, S):
    """against f64 the outputs are off by their own rounding to bf16 and no more: 2^-8 / sqrt(3) of a unit whose values lie
    log-uniform in it, 1.66e-3 in the relative 2-norm, and a twentieth over that; weights rounded once to bf16 against a
    batch's maximum make it 2.1e-3"""
    D = 128
    cap = n0 + T + 30
    g = torch.Generator(device="cuda").manual_seed(1400 + n0 + T)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    K, V, q = rnd(Hk, cap, D), rnd(Hk, cap, D), rnd(T, Hq * D)
    n0t = torch.tensor([n0], dtype=torch.int32, device="cuda")
    scratch = card.attn_scratch(T, Hq, Hk, D, S)
    att = torch.zeros(T, Hq * D, dtype=torch.bfloat16, device="cuda")
    scale = 1.0 / np.sqrt(D)
    if T == 1:  # no norm, and a rope that leaves q and k as they are
        cos, sin = torch.ones(cap, D, device="cuda").to(torch.bfloat16), torch.zeros(cap, D, device="cuda").to(torch.bfloat16)
        qkv = torch.cat([q[0], rnd(2 * Hk * D)])[None]
        card.attn_decode_qkv_span(qkv, None, None, 1e-6, cos, sin, n0t, K, V, att, Hq, Hk, D, scale, S, scratch)
    else:
        card.attn_decode(q, K, V, att, n0t, Hq, Hk, D, scale, S, scratch)
    ref = torch.empty(T, Hq, D, dtype=torch.float64, device="cuda")
    hidden = torch.ones(T, n0 + T, dtype=torch.bool, device="cuda").triu(n0 + 1)
    for h in range(Hq):
        k, v = K[h // (Hq // Hk), : n0 + T].double(), V[h // (Hq // Hk), : n0 + T].double()
        s = (q.view(T, Hq, D)[:, h].double() @ k.t()) * scale
        ref[:, h] = torch.softmax(s.masked_fill(hidden, float("-inf")), 1) @ v
    off = float((att.double() - ref.view(T, -1)).norm() / ref.norm())
    assert off <= 1.05 * 1.66e-3, off


@pytest.mark.parametrize("n0,T,Hq,Hk,S", [(1000, 20, 8, 8, 2), (700, 17, 32, 8, 1), (300, 5, 16, 2, 1), (520, 20, 8, 2, 5)])
def test_values_that_are_not_finite(card, n0, T, Hq, Hk, S):
    """an infinite or NaN value every row sees: an output is what the vector kernels make of it - the same infinity, NaN
    where they are NaN -, and the other outputs are finite and what they would be"""
    D = 128
    cap = n0 + T + 30
    g = gen(1500 + n0 + T)
    K = torch.randn(Hk, cap, D, generator=g).to(torch.bfloat16).cuda()
    V = torch.randn(Hk, cap, D, generator=g).to(torch.bfloat16)
    for slot, dim, v in ((17, 3, "inf"), (n0 - 1, 5, "-inf"), (130, 7, "nan"), (20, 9, "inf"), (21, 9, "-inf")):
        V[0, slot, dim] = float(v)
    V = V.cuda()
    q = torch.randn(T, Hq * D, generator=g).to(torch.bfloat16).cuda()
    par = torch.arange(-1, T - 1, dtype=torch.int32, device="cuda")
    n0t = torch.tensor([n0], dtype=torch.int32, device="cuda")
    scratch = card.attn_scratch(T, Hq, Hk, D, S)

    def run(knob):
        att = torch.zeros(T, Hq * D, dtype=torch.bfloat16, device="cuda")
        card.set_tuning("attn_mfma", knob)
        try:
            card.attn_decode(q, K, V, att, n0t, Hq, Hk, D, 1.0 / np.sqrt(D), S, scratch, par=par)
        finally:
            card.set_tuning("attn_mfma", -1)
        return att.float()

    want, got = run(0), run(-1)
    assert torch.equal(torch.isnan(want), torch.isnan(got)) and int(torch.isnan(want).sum()) == T * (Hq // Hk) * 2
    assert torch.equal(want[want.isinf()], got[want.isinf()]) and int(want.isinf().sum()) == T * (Hq // Hk) * 2
    fin = torch.isfinite(want)
    assert bool(torch.isfinite(got[fin]).all())
    assert float((want[fin] - got[fin]).abs().max()) <= float(want[fin].abs().max()) * 2.0**-7


# a chain without a tree and a tree; the pass's own rows within a batch and across two; several workgroups a kv head
@pytest.mark.parametrize("n0,T,Hq,Hk,S,tree", [(1000, 3, 8, 2, 2, False), (300, 9, 8, 8, 1, False), (250, 17, 32, 8, 1, False),
                                               (300, 20, 16, 2, 1, False), (300, 33, 8, 8, 1, False), (120, 12, 16, 2, 1, True)])
@pytest.mark.parametrize("what", ["inf", "nan"])
def test_a_later_row_never_reaches_an_earlier_one(card, n0, T, Hq, Hk, S, tree, what):
    """the last row's k and v not finite - a padding row, or one that overflowed: the rows that do not see it keep their
    bits"""
    D = 128
    cap = n0 + T + 30
    g = gen(1600 + n0 + T)
    K = torch.randn(Hk, cap, D, generator=g).to(torch.bfloat16).cuda()
    V = torch.randn(Hk, cap, D, generator=g).to(torch.bfloat16).cuda()
    q = torch.randn(T, Hq * D, generator=g).to(torch.bfloat16).cuda()
    par = torch.tensor([-1] + [0] * (T - 1), dtype=torch.int32, device="cuda") if tree else None
    n0t = torch.tensor([n0], dtype=torch.int32, device="cuda")
    scratch = card.attn_scratch(T, Hq, Hk, D, S)

    def run():
        att = torch.zeros(T, Hq * D, dtype=torch.bfloat16, device="cuda")
        card.attn_decode(q, K, V, att, n0t, Hq, Hk, D, 1.0 / np.sqrt(D), S, scratch, par=par)
        return att

    want = run()
    V[:, n0 + T - 1] = float(what)
    K[:, n0 + T - 1] = float(what)
    got = run()
    assert torch.equal(got[: T - 1], want[: T - 1])
    assert not bool(torch.isfinite(got[T - 1].float()).any())


# windows shorter than the path, of a power of two and around it, as long as the pass; whole spans and the first batches of
# one before every row's window; deep and bushy trees and a chain; both matrix-core kernels (spans of 128 keys: one batch)
@pytest.mark.parametrize("n0,T,Hq,Hk,S,shape,win", [
    (900, 32, 8, 8, 2, "deep", 1), (900, 32, 8, 8, 2, "deep", 7), (900, 32, 16, 2, 1, "deep", 31), (900, 32, 8, 2, 3, "deep", 32),
    (900, 32, 8, 2, 3, "deep", 33), (700, 20, 32, 8, 2, "bushy", 4), (700, 9, 8, 8, 6, "bushy", 130), (700, 9, 8, 2, 6, "deep", 16),
    (900, 40, 8, 8, 2, None, 5), (900, 17, 32, 8, 8, None, 200), (20, 6, 8, 1, 1, "deep", 3)])
def test_windows_over_trees(card, n0, T, Hq, Hk, S, shape, win):
    D = 128
    cap = n0 + T + 60
    span = -(-(-(-cap // S)) // 128) * 128
    g = gen(1700 + n0 + T + win)
    K = torch.randn(Hk, cap, D, generator=g).to(torch.bfloat16)
    V = torch.randn(Hk, cap, D, generator=g).to(torch.bfloat16)
    q = (2 * torch.randn(T, Hq * D, generator=g)).to(torch.bfloat16)
    par = None
    if shape == "deep":  # a long path with a leaf beside every fifth row
        par = [-1] + [t - 2 if t % 5 == 4 else t - 1 for t in range(1, T)]
        par = [p if p < 0 or p % 5 != 4 else p - 1 for p in par]
    elif shape == "bushy":
        par = [-1] + [int(torch.randint(-1, t, (1,), generator=g)) for t in range(1, T)]
    seen = [seen_by(t, n0, par, win) for t in range(T)]
    first = min(min(s) for s in seen)
    if span > 128:  # slots that the window has left behind, and what lies past the pass, hold anything
        K[:, :first], V[:, :first] = float("nan"), float("nan")
    K[:, n0 + T:], V[:, n0 + T:] = float("nan"), float("nan")
    part = None if par is None else torch.tensor(par, dtype=torch.int32, device="cuda")
    scale = 1.0 / np.sqrt(D)
    att = torch.zeros(T, Hq * D, dtype=torch.bfloat16, device="cuda")
    card.attn_decode(q.cuda(), K.cuda(), V.cuda(), att, torch.tensor([n0], dtype=torch.int32, device="cuda"), Hq, Hk, D,
                     scale, S, card.attn_scratch(T, Hq, Hk, D, S), par=part, win=win)
    got = att.float().cpu().numpy()
    for t in range(T):
        want = od.attention(q[t].float().numpy().reshape(Hq, D), K[:, seen[t]].float().numpy(),
                            V[:, seen[t]].float().numpy(), scale)
        worst = np.abs(got[t].reshape(Hq, D) - want).max() / np.abs(want).max()
        assert worst <= 2.0**-7, (t, worst)  # weights and outputs in bf16, as above


@pytest.mark.parametrize("n0,T,Hq,Hk,S,tree", [(2100, 16, 32, 8, 16, False), (3000, 21, 16, 2, 23, True), (2100, 17, 16, 8, 12, True)])
def test_a_workgroups_tiles_change_no_bit(card, n0, T, Hq, Hk, S, tree):
    """a kv head's rows in workgroups of two tiles of pairs (all the kv heads: more workgroups of one than CUs) and of one (the
    kv head by itself)"""
    D, G = 128, Hq // Hk
    cap = n0 + T + 30
    g = gen(1900 + n0 + T)
    K = torch.randn(Hk, cap, D, generator=g).to(torch.bfloat16).cuda()
    V = torch.randn(Hk, cap, D, generator=g).to(torch.bfloat16).cuda()
    q = torch.randn(T, Hk, G * D, generator=g).to(torch.bfloat16).cuda()
    par = [-1] + [int(torch.randint(-1, t, (1,), generator=g)) for t in range(1, T)] if tree else None
    part = None if par is None else torch.tensor(par, dtype=torch.int32, device="cuda")
    n0t = torch.tensor([n0], dtype=torch.int32, device="cuda")

    def run(q, K, V, heads, kv_heads):
        att = torch.zeros(T, heads * D, dtype=torch.bfloat16, device="cuda")
        card.attn_decode(q.reshape(T, -1), K, V, att, n0t, heads, kv_heads, D, 1.0 / np.sqrt(D), S,
                         card.attn_scratch(T, heads, kv_heads, D, S), par=part)
        return att

    both = run(q, K, V, Hq, Hk).view(T, Hk, G * D)
    for h in range(0, Hk, max(1, Hk - 1) if G > 2 else Hk):
        if G > 2:  # with two heads a kv head so few workgroups stay with the vector kernels
            assert torch.equal(run(q[:, h].contiguous(), K[h : h + 1], V[h : h + 1], G, 1), both[:, h])
    if G <= 2:
        half = Hk // 2
        part_of = run(q[:, :half].contiguous(), K[:half], V[:half], Hq // 2, half).view(T, half, G * D)
        assert torch.equal(part_of, both[:, :half])


# a cache of 9000 slots with few keys, one batch and the first of the next, as many as the spans take in one batch each and
# one more, the last slot; 32 spans (a workgroup a CU), 7 and 1
@pytest.mark.parametrize("n0", [0, 1, 127, 128, 4094, 4095, 4096, 8999])
@pytest.mark.parametrize("Hq,Hk,S", [(32, 8, 32), (16, 2, 7), (4, 2, 1)])
def test_one_row_over_the_keys_there_are(card, n0, Hq, Hk, S):
    """`attn_decode_qkv_span` at one row cuts its spans from the keys the cache holds: against f64 attention, the row in its
    slot and nothing else in the cache touched, whatever the empty slots hold"""
    D, cap = 128, 9000
    g = torch.Generator(device="cuda").manual_seed(1800 + n0)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    K, V, qkv = rnd(Hk, cap, D), rnd(Hk, cap, D), rnd(1, (Hq + 2 * Hk) * D)
    K[:, n0:], V[:, n0:] = float("nan"), float("nan")
    K0, V0 = K.clone(), V.clone()
    cos, sin = torch.ones(cap, D, device="cuda").to(torch.bfloat16), torch.zeros(cap, D, device="cuda").to(torch.bfloat16)
    att = torch.zeros(1, Hq * D, dtype=torch.bfloat16, device="cuda")
    card.attn_decode_qkv_span(qkv, None, None, 1e-6, cos, sin, torch.tensor([n0], dtype=torch.int32, device="cuda"), K, V,
                              att, Hq, Hk, D, 1.0 / np.sqrt(D), S, card.attn_scratch(1, Hq, Hk, D, S))
    rows = qkv[0].view(Hq + 2 * Hk, D)
    K0[:, n0], V0[:, n0] = rows[Hq : Hq + Hk], rows[Hq + Hk :]
    for a, b in ((K, K0), (V, V0)):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    for h in range(Hq):
        k, v = K[h // (Hq // Hk), : n0 + 1].double(), V[h // (Hq // Hk), : n0 + 1].double()
        want = torch.softmax((k @ rows[h].double()) / np.sqrt(D), 0) @ v
        off = float((att.view(Hq, D)[h].double() - want).norm() / want.norm())
        assert off <= 2.0**-8, (h, off)  # the outputs' rounding to bf16
