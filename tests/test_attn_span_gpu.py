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
