"""A routed layer keeps no buffer between its calls: what one call's gate / up launch writes for its down launch belongs to that
call, so calls on two streams do not meet in it and a recorded graph's addresses stay its own."""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from btb_amd.moe import Experts, MxExpertsLayer
from btb_amd.native import HipCard

from .helpers import acts_bf16, gen


class Recorder:
    """a card that keeps the buffer each call is handed"""

    def __init__(self) -> None:
        self.buffers: list[torch.Tensor | None] = []

    def moe_experts(self, gate_up, down, x, idx, w, y=None, gu=None):
        self.buffers.append(gu)
        return x

    def moe_experts_mx4(self, ex, x, idx, w, y=None, h=None, oss=True, alpha=1.702, limit=7.0):
        self.buffers.append(h)
        return x


@pytest.mark.parametrize("form", ["bf16", "mxfp4"])
def test_no_buffer_is_shared_between_calls(form):
    card = Recorder()
    if form == "bf16":
        layer = Experts(card, torch.zeros(4, 64, 32, dtype=torch.bfloat16), torch.zeros(4, 32, 32, dtype=torch.bfloat16))
    else:
        layer = MxExpertsLayer(card, SimpleNamespace(experts=4, hidden=32, intermediate=32, gate_up_bias=None, down_bias=None), oss=False)
    for T in (2, 1, 2, 5, 2):
        layer(torch.zeros(T, 32, dtype=torch.bfloat16), torch.zeros(T, 2, dtype=torch.int64), torch.zeros(T, 2))
    held = [b for b in card.buffers if b is not None]
    places = [b.untyped_storage().data_ptr() for b in held]
    assert len(set(places)) == len(places)


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["bf16", "mxfp4"])
def test_a_recorded_layer_outlives_wider_eager_calls(card: HipCard, form):
    """two rows recorded, then sixteen rows and another k run eagerly and memory of those sizes taken: every replay gives the
    recorded call's values and leaves that memory alone"""
    from btb_amd import mxfp4
    from btb_amd.load import MxExperts

    E, H, I, g = 8, 256, 128, gen(77)
    gu, dn = ((torch.randn(E, r, c, generator=g) * 0.05) for r, c in ((2 * I, H), (H, I)))
    if form == "bf16":
        layer = Experts(card, gu.to(torch.bfloat16).cuda(), dn.to(torch.bfloat16).cuda())
    else:
        (gb, gs), (db, ds) = mxfp4.quantize(gu.reshape(-1, H)), mxfp4.quantize(dn.reshape(-1, I))
        stacks = MxExperts(gb.reshape(E, 2 * I, H // 32, 16).cuda(), gs.reshape(E, 2 * I, H // 32).cuda(),
                           db.reshape(E, H, I // 32, 16).cuda(), ds.reshape(E, H, I // 32).cuda(), None, None)
        layer = MxExpertsLayer(card, stacks, oss=False)

    def call_of(T, k):
        picks = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(torch.int32).cuda()
        return acts_bf16(T, H, seed=78 + T).cuda(), picks, torch.rand(T, k, generator=g).to(torch.bfloat16).cuda()

    two, wide = call_of(2, 2), call_of(16, 4)
    want, want_wide = layer(*two).clone(), layer(*wide).clone()
    out = torch.empty_like(want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        layer(*two, out)
    for _ in range(3):
        assert torch.equal(layer(*wide), want_wide)
        guard = [torch.full((n,), 3.0, dtype=torch.bfloat16, device="cuda") for n in (2 * 2 * I, 2 * 2 * 2 * I, 16 * 4 * 2 * I)]
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and all(bool((t == 3.0).all()) for t in guard)
