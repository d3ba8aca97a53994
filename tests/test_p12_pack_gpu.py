"""The 12-bit packer on the card (`HipCard.p12_pack`, `P12Weight.pack`) against the oracle's packer, byte for byte, at the
sizes where its pieces meet: a lane's 8 weights, a chunk of 2048, a workgroup's 32768, rows that begin inside a chunk, odd
tails; and on values with no escapes, with few and with most weights escaped."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from btb_amd.pack12 import P12Weight, pack_bf16
from oracle import codecs

from .helpers import bits16

pytestmark = pytest.mark.gpu


def values(kind: str, n: int) -> torch.Tensor:
    g = torch.Generator().manual_seed(0x0B7B + n)
    if kind == "normal":
        return (torch.randn(n, generator=g) * 0.02).to(torch.bfloat16)
    if kind == "bits":  # every bit pattern: 15 high bytes of 256 have a code
        return torch.randint(-(2**15), 2**15, (n,), generator=g).to(torch.int16).view(torch.bfloat16)
    return torch.full((n,), -1.5, dtype=torch.bfloat16)


@pytest.mark.parametrize("kind", ["normal", "bits", "one"])
@pytest.mark.parametrize("rows,cols", [(1, 1), (1, 7), (3, 5), (2, 8), (7, 33), (16, 128), (17, 121), (1, 2047), (1, 32768),
                                       (3, 10923), (257, 130), (40, 2560), (5, 9728), (300, 1000)])
def test_packed_on_the_card(card, kind, rows, cols):
    w = values(kind, rows * cols).reshape(rows, cols)
    pw = P12Weight.pack(w.cuda(), card)
    lo, hi4, table, idx, val = codecs.pack12_pack(bits16(w))
    for got, want in ((pw.lo, lo), (pw.hi4, hi4), (pw.table, table), (pw.esc_idx, idx), (pw.esc_val, val)):
        assert np.array_equal(got.cpu().numpy(), want)
    # what the constructor makes at upload of a stored matrix's arrays
    up = P12Weight(*(t.cuda() for t in pack_bf16(w)), rows, cols, card)
    for name in ("pairs", "row_ptr", "row_esc"):
        a, b = getattr(pw, name), getattr(up, name)
        assert (a is None and b is None and cols > 32767) or torch.equal(a, b), name
    assert np.array_equal(pw.row_ptr.cpu().numpy(), np.searchsorted(idx, np.arange(rows + 1) * cols))


@pytest.mark.parametrize("crowd", [63, 64, 65, 300])
@pytest.mark.parametrize("cols", [2560, 1000, 7, 40000])
def test_escapes_in_crowds(card, crowd, cols):
    """The encoder lists up to 64 escapes a wave (8192 weights); a workgroup (32768) where a wave has more is read out of its
    codes: crowds of that many, as they begin and end a wave's and a workgroup's weights, beside workgroups that have few."""
    rows = -(-5 * 32768 // cols)
    i = torch.arange(rows * cols, dtype=torch.int32)
    w = ((0x30 + i % 15) << 8) | (i % 251)  # fifteen high bytes fill the table, every other is an escape
    for at in (8192 - 10, 32768 + 8192, 3 * 32768 - crowd, 4 * 32768 - 3):
        w[at : at + crowd] = 0x7100 + torch.arange(crowd, dtype=torch.int32) % 256
    w[5::20011] = 0x7201
    w = w.to(torch.int16).view(torch.bfloat16)
    w = w.reshape(rows, cols)
    pw = P12Weight.pack(w.cuda(), card)
    lo, hi4, table, idx, val = codecs.pack12_pack(bits16(w))
    assert idx.size >= 4 * crowd and (np.bincount(idx // 8192) >= crowd).any()
    for got, want in ((pw.lo, lo), (pw.hi4, hi4), (pw.table, table), (pw.esc_idx, idx), (pw.esc_val, val)):
        assert np.array_equal(got.cpu().numpy(), want)
    assert np.array_equal(pw.row_ptr.cpu().numpy(), np.searchsorted(idx, np.arange(rows + 1) * cols))


def test_a_view_that_is_not_16_byte_aligned(card):
    w = values("normal", 4096 + 3)
    pw = P12Weight.pack(w.cuda()[3:].reshape(64, 64), card)
    lo, hi4, _, idx, _ = codecs.pack12_pack(bits16(w[3:]))
    assert np.array_equal(pw.lo.cpu().numpy(), lo) and np.array_equal(pw.hi4.cpu().numpy(), hi4)
    assert np.array_equal(pw.esc_idx.cpu().numpy(), idx)


def test_the_rows_words_of_the_tallest_matrices(card):
    """more rows than a launch has threads for their words: one column, 2^29 + 3 rows, an escape in the first and the last"""
    rows = 2**29 + 3
    lo = torch.full((rows,), 7, dtype=torch.uint8, device="cuda")
    idx = torch.tensor([0, rows - 1], dtype=torch.int32, device="cuda")
    val = torch.tensor([0x41, 0x42], dtype=torch.uint8, device="cuda")
    row_ptr = torch.ones(rows + 1, dtype=torch.int32, device="cuda")
    row_ptr[0], row_ptr[-1] = 0, 2
    words = card.p12_row_esc(lo, idx, val, row_ptr, rows, 1)
    none = 0x7FFF << 16
    assert words[0].tolist() == [7 | 0x41 << 8] + [none] * 7 and words[-1].tolist() == [7 | 0x42 << 8] + [none] * 7
    for part in words[1:-1].split(2**27):
        assert int(part.min()) == none and int(part.max()) == none
