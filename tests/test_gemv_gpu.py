"""The bf16 decode matvec on the GPU (through the C ABI) against the CPU oracle on the same seeded inputs.

Bar: max |y_gpu - y_ref| / max |y_ref| <= 1e-2 on the bf16 outputs, y_ref the oracle's f32
result rounded to bf16. Both sides accumulate in f32 with one fused multiply-add per weight; they differ only in the
order of the additions (<= ~sqrt(C) * 2^-24 relative to sum |w x|, far below a bf16 ulp), so what is seen is at most a
bf16 rounding flip: 2^-8 relative to the output. The reference's own card bar, one bf16 ulp of the largest output
(tests/kernels/test_card_kernels.py:135-148), is asserted too.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

import oracle
from oracle import codecs

from .helpers import acts_bf16, bits16, weights_bf16

pytestmark = pytest.mark.gpu

REL_TOL = 1e-2


def oracle_bf16_out(w: torch.Tensor, x: torch.Tensor) -> np.ndarray:
    """the CPU path's answer as the card stores it: f32 lane sums, rounded to bf16 (kept as f32)"""
    y = oracle.gemv_bf16(bits16(w), x.float().numpy(), threads=0)
    return codecs.round_bf16(y)


def check(y: torch.Tensor, ref: np.ndarray) -> None:
    got = y.float().cpu().numpy()
    peak = np.abs(ref).max()
    err = np.abs(got - ref).max()
    assert err <= REL_TOL * peak, (err, peak)
    assert err <= peak * 2.0**-7, (err, peak)


@pytest.mark.parametrize("R,C", [(9728, 2560), (2560, 9728), (6144, 2560), (2560, 4096), (2048, 768), (1536, 2048),
                                 (128, 2048), (1000, 264), (7, 8), (3, 1032)])
@pytest.mark.parametrize("M", [1, 4])
def test_gemv_bf16_matches_oracle(card, R, C, M):
    w = weights_bf16(R, C, seed=100)
    x = acts_bf16(M, C, seed=101)
    y = card.gemv(w.cuda(), x.cuda())
    check(y, oracle_bf16_out(w, x))


@pytest.mark.parametrize("M", [2, 3, 4, 5, 7])
def test_row_of_a_wide_pass_is_its_one_row_pass(card, M):
    """native/cuda/btb_kernels.cu:84-88 and tests/kernels/test_card_kernels.py:145-148: row m does not depend on M"""
    R, C = 2560, 4096
    w = weights_bf16(R, C, seed=110).cuda()
    x = acts_bf16(M, C, seed=111).cuda()
    y = card.gemv(w, x)
    check(y, oracle_bf16_out(w.cpu(), x.cpu()))
    for m in (0, M - 1):
        solo = card.gemv(w, x[m : m + 1].contiguous())
        assert torch.equal(solo[0].view(torch.int16), y[m].view(torch.int16))


@pytest.mark.parametrize("R,C", [(2560, 9728), (2561, 5128), (7, 10240), (1, 6152), (5000, 8192), (3000, 9736)])
def test_long_rows_by_two_waves(card, R, C):
    """rows of 5121 .. 10240 values are summed by two waves, a half each (`gemv_halves`): against the oracle at one to
    four rows of x; row m of a pass is its one-row pass bit for bit; the add + norm in the x load gives the bits of
    add_rmsnorm followed by the plain matvec, the gate / up fold those of the plain matvec followed by silu_mul; with
    the split switched off (knob gemv_halves = 0: the whole-row kernel,
    another order of summation) the outputs stay within one bf16 ulp of the largest. Shapes: the down projection, odd
    row counts, the shortest and the longest row the split takes, rows of an odd number of units, and a matrix tall
    enough that workgroups take several turns."""
    w = weights_bf16(R, C, seed=120)
    x = acts_bf16(4, C, seed=121)
    ref = oracle_bf16_out(w, x)
    wd, xd = w.cuda(), x.cuda()
    y4 = card.gemv(wd, xd)
    check(y4, ref)
    for M in (1, 2, 3):
        ym = card.gemv(wd, xd[:M].contiguous())
        assert torch.equal(ym.view(torch.int16), y4[:M].view(torch.int16)), M
    solo = card.gemv(wd, xd[3:4].contiguous())
    assert torch.equal(solo[0].view(torch.int16), y4[3].view(torch.int16))
    # the add + norm form (workgroups of four waves) against the two launches (ten waves): the same bits
    for M in (1, 3):
        h = acts_bf16(M, C, seed=122).cuda()
        d = acts_bf16(M, C, seed=123).cuda()
        nw = (1.0 + 0.1 * torch.randn(C, generator=torch.Generator().manual_seed(124))).to(torch.bfloat16).cuda()
        h1, x1 = h.clone(), torch.empty_like(h)
        card.add_rmsnorm(h1, d, nw, 1e-6, x1)
        want = card.gemv(wd, x1)
        h2 = torch.empty_like(h)
        out = torch.empty(M, R, dtype=torch.bfloat16, device="cuda")
        card.gemv_norm(wd, h, d, nw, 1e-6, h2, out, glu=False)
        assert torch.equal(out.view(torch.int16), want.view(torch.int16))
        assert torch.equal(h2.view(torch.int16), h1.view(torch.int16))
    # the gate / up fold over such rows (four waves an output): the plain matvec, then silu_mul, bit for bit
    if R % 2 == 0:
        for M in (1, 3):
            xm = xd[:M].contiguous()
            want = torch.empty(M, R // 2, dtype=torch.bfloat16, device="cuda")
            card.silu_mul(card.gemv(wd, xm), want)
            got = card.gemv_glu_silu(wd, xm)
            assert torch.equal(got.view(torch.int16), want.view(torch.int16)), M
    card.set_tuning("gemv_halves", 0)
    try:
        whole = card.gemv(wd, xd)
    finally:
        card.set_tuning("gemv_halves", -1)
    check(whole, ref)
    peak = float(np.abs(ref).max())
    assert float((whole.float() - y4.float()).abs().max()) <= peak * 2.0**-7


def test_long_rows_by_two_waves_over_drawn_shapes(card):
    """twenty drawn shapes in and around the split's range of row lengths (any multiple of 8 from 5000 to 10400 values,
    1 .. 3000 rows, 1 .. 4 rows of x): the oracle's bar, and every row of the pass the bits of its one-row pass"""
    rng = np.random.default_rng(20261)
    for i in range(20):
        R = int(rng.integers(1, 3001))
        C = 8 * int(rng.integers(625, 1301))
        M = int(rng.integers(1, 5))
        w = weights_bf16(R, C, seed=2000 + i)
        x = acts_bf16(M, C, seed=3000 + i)
        wd, xd = w.cuda(), x.cuda()
        y = card.gemv(wd, xd)
        check(y, oracle_bf16_out(w, x))
        for m in range(M):
            solo = card.gemv(wd, xd[m : m + 1].contiguous())
            assert torch.equal(solo[0].view(torch.int16), y[m].view(torch.int16)), (R, C, M, m)


@pytest.mark.parametrize("R,C", [(9728, 2560), (2560, 9728), (2560, 4096), (1000, 96), (18, 32)])
@pytest.mark.parametrize("M", [8, 16, 32, 12, 40])
def test_verify_widths_on_the_matrix_cores(card, R, C, M):
    """M >= 8 runs on MFMA: within the oracle's bar, and a row's bits are the same at every verify width (the
    reference's tensor-core matvec keeps that law within its family: tests/kernels/test_card_kernels.py:513-524)"""
    w = weights_bf16(R, C, seed=112).cuda()
    x = acts_bf16(M, C, seed=113).cuda()
    y = card.gemv(w, x)
    check(y, oracle_bf16_out(w.cpu(), x.cpu()))
    y8 = card.gemv(w, x[:8].contiguous())
    assert torch.equal(y8.view(torch.int16), y[:8].view(torch.int16))
    # the vector-ALU form of the same pass agrees to the same bar and equals the one-row pass bit for bit
    card.set_tuning("gemv_no_mfma", 1)
    try:
        v = card.gemv(w, x)
        solo = card.gemv(w, x[M - 1 :].contiguous())
    finally:
        card.set_tuning("gemv_no_mfma", -1)
    check(v, oracle_bf16_out(w.cpu(), x.cpu()))
    assert torch.equal(solo[0].view(torch.int16), v[M - 1].view(torch.int16))


def test_repeat_runs_are_bit_stable(card):
    w = weights_bf16(9728, 2560, seed=120).cuda()
    x = acts_bf16(1, 2560, seed=121).cuda()
    a = card.gemv(w, x).clone()
    for _ in range(5):
        assert torch.equal(card.gemv(w, x).view(torch.int16), a.view(torch.int16))


@pytest.mark.parametrize("M", [1, 4])
def test_silu_fold_equals_two_steps(card, M):
    """tests/kernels/test_card_kernels.py:376-391: the folded down projection equals act-mul then the plain matvec"""
    R, C = 2560, 9728
    w = weights_bf16(R, C, seed=130).cuda()
    gu = acts_bf16(M, 2 * C, seed=131).cuda()
    g, u = gu[:, :C].float(), gu[:, C:].float()
    s = (g / (1 + torch.exp(-g))).to(torch.bfloat16).float()
    x = (s * u).to(torch.bfloat16)
    folded = card.gemv_silu(w, gu)
    plain = card.gemv(w, x.contiguous())
    # the activation's exp may differ from torch's in the last bit, which can flip a bf16 rounding of x here and there
    ref = oracle_bf16_out(w.cpu(), x.cpu())
    check(folded, ref)
    frac = (folded != plain).float().mean().item()
    assert frac < 0.02, frac


@pytest.mark.parametrize("I,C", [(9728, 2560), (768, 2048), (96, 4096), (64, 9728), (40, 64)])
@pytest.mark.parametrize("M", [8, 16, 24])
def test_glu_kernel_at_the_verify_widths(card, I, C, M):
    """gate, up and the activation in the matrix-core kernel: the bits of its matvec followed by silu_mul, for each of
    the kernel's forms (and the vector passes where I is no multiple of 16)"""
    w = weights_bf16(2 * I, C, seed=152).cuda()
    x = acts_bf16(M, C, seed=153).cuda()
    gu = card.gemv(w, x)
    want = torch.empty(M, I, dtype=torch.bfloat16, device="cuda")
    card.silu_mul(gu, want)
    got = card.gemv_glu_silu(w, x)
    if I % 16 == 0:
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    else:  # vector passes against a matrix-core matvec: the bar, not the bits
        assert float((got.float() - want.float()).abs().max()) <= 2.0**-7 * float(want.float().abs().max())


@pytest.mark.parametrize("M", [1, 3])
def test_glu_kernel_equals_matvec_then_silu_mul(card, M):
    I, C = 9728, 2560
    w = weights_bf16(2 * I, C, seed=150).cuda()
    x = acts_bf16(M, C, seed=151).cuda()
    gu = card.gemv(w, x)
    want = torch.empty(M, I, dtype=torch.bfloat16, device="cuda")
    card.silu_mul(gu, want)
    got = card.gemv_glu_silu(w, x)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("M,with_y,glu,C", [(1, True, False, 2560), (1, False, False, 2560), (2, True, True, 2560),
                                              (1, True, True, 2560), (5, True, False, 2560), (8, True, True, 2560),
                                              (8, False, False, 2560), (16, True, True, 2560), (13, True, False, 2560),
                                              (7, True, True, 2048), (16, True, False, 1536), (4, True, False, 1280),
                                              (17, True, False, 2560), (35, True, True, 2560)])
def test_norm_folded_into_the_x_load_changes_no_bit(card, M, with_y, glu, C):
    """the residual add + norm made by the matvec itself (the vector kernels up to four rows a pass; from five rows
    the matrix cores, where the kernel makes the rows for rows of 1312 .. 2560 values, 16 rows a launch) against
    add_rmsnorm followed by the matvec: the same output and the same new residual, bit for bit"""
    R = 6144
    w = weights_bf16(R, C, seed=160).cuda()
    h = acts_bf16(M, C, seed=161).cuda()
    y = acts_bf16(M, C, seed=162).cuda() if with_y else None
    nw = (1.0 + 0.1 * torch.randn(C, generator=torch.Generator().manual_seed(163))).to(torch.bfloat16).cuda()
    h1, x1 = h.clone(), torch.empty_like(h)
    card.add_rmsnorm(h1, y, nw, 1e-6, x1)
    want = card.gemv_glu_silu(w, x1) if glu else card.gemv(w, x1)
    h2 = torch.empty_like(h)
    out = torch.empty(M, R // 2 if glu else R, dtype=torch.bfloat16, device="cuda")
    card.gemv_norm(w, h, y, nw, 1e-6, h2, out, glu=glu)
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
    assert torch.equal(h2.view(torch.int16), h1.view(torch.int16))
    with pytest.raises(ValueError):
        card.gemv_norm(w, h, y, nw, 1e-6, h, out, glu=glu)


@pytest.mark.parametrize("M", [1, 3, 8, 16])
def test_embedding_rows_gathered_by_the_first_matvec(card, M):
    """`gemv_embed_norm` against embed + add_rmsnorm + gemv: the same output and residual rows, ids outside the table
    clamped into it - on the vector kernels and, from five rows, on the matrix cores"""
    R, C, vocab = 4096, 2560, 300
    w = weights_bf16(R, C, seed=170).cuda()
    table = acts_bf16(vocab, C, seed=171).cuda()
    nw = (1.0 + 0.1 * torch.randn(C, generator=torch.Generator().manual_seed(172))).to(torch.bfloat16).cuda()
    ids = torch.randint(0, vocab, (M,), generator=torch.Generator().manual_seed(173), dtype=torch.int32)
    ids[0] = vocab + 5
    ids = ids.cuda()
    h1 = torch.empty(M, C, dtype=torch.bfloat16, device="cuda")
    card.embed(table, ids, h1)
    x1 = torch.empty_like(h1)
    card.add_rmsnorm(h1, None, nw, 1e-6, x1)
    want = card.gemv(w, x1)
    h2 = torch.empty_like(h1)
    out = torch.empty(M, R, dtype=torch.bfloat16, device="cuda")
    card.gemv_embed_norm(w, table, ids, nw, 1e-6, h2, out)
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
    assert torch.equal(h2.view(torch.int16), h1.view(torch.int16))


def test_rows_a_tile_change_no_bit_over_drawn_shapes(card):
    """the matrix-core matvec takes tiles of twelve or ten rows where sixteen would leave CUs idle (knob mfma_tile_rows
    = 0: always sixteen): over thirty drawn shapes - any multiple of 16 rows, the row lengths of the kernel's classes,
    5 .. 32 rows of x - the same bits either way, within the bar of an f32 product"""
    rng = np.random.default_rng(20252)
    lower = 0
    for _ in range(30):
        R = 16 * int(rng.integers(1, 700))
        C = int(rng.choice([2560, 4096, 1536, 5120, 9728, 7168]))
        M = int(rng.integers(5, 33))
        w = weights_bf16(R, C, seed=int(rng.integers(1 << 30))).cuda()
        x = acts_bf16(M, C, seed=int(rng.integers(1 << 30))).cuda()
        y = card.gemv(w, x)
        card.set_tuning("mfma_tile_rows", 0)
        try:
            y16 = card.gemv(w, x)
        finally:
            card.set_tuning("mfma_tile_rows", -1)
        assert torch.equal(y.view(torch.int16), y16.view(torch.int16)), (R, C, M)
        ref = x.float() @ w.float().t()
        assert float((y.float() - ref).abs().max()) <= 2.0**-7 * float(ref.abs().max()), (R, C, M)
        lower += int(R % 12 == 0 or R % 10 == 0)
    assert lower >= 5  # the draw holds row counts the lower tiles apply to


def test_refusals_launch_nothing(card):
    w = weights_bf16(16, 64, seed=140).cuda()
    x = acts_bf16(1, 64, seed=141).cuda()
    with pytest.raises(ValueError):
        card.gemv(w.float(), x)
    with pytest.raises(ValueError):
        card.gemv(w, x.cpu())
    with pytest.raises(ValueError):
        card.gemv(w, x, torch.empty(3, dtype=torch.bfloat16, device="cuda"))
    L = card.lib
    y = torch.full((1, 16), 7.0, dtype=torch.bfloat16, device="cuda")
    assert L.btb_hip_gemv_bf16(None, card.ptr(ctypes.c_void_p, x), card.ptr(ctypes.c_void_p, y), 16, 64, 1, None) == -1
    assert L.btb_hip_gemv_bf16(card.ptr(ctypes.c_void_p, w), card.ptr(ctypes.c_void_p, x), card.ptr(ctypes.c_void_p, y), 0, 64, 1, None) == -6
    assert L.btb_hip_gemv_bf16(card.ptr(ctypes.c_void_p, w), card.ptr(ctypes.c_void_p, x), card.ptr(ctypes.c_void_p, y), 16, 60, 1, None) == -6  # C % 8
    assert L.btb_hip_gemv_bf16(None, card.ptr(ctypes.c_void_p, x), card.ptr(ctypes.c_void_p, y), 0, 64, 1, None) == -1  # null before domain
    torch.cuda.synchronize()
    assert torch.all(y == 7.0)


@pytest.mark.parametrize("R,C", [(16, 1312), (17, 2592), (33, 2560), (100, 3008), (520, 9728), (1001, 4096), (2560, 9728),
                                 (4112, 10240), (2064, 7168)])
@pytest.mark.parametrize("M", [5, 8, 16, 17, 31, 32, 33, 50])
def test_columns_split_over_workgroups_change_no_bit(card, R, C, M):
    """The wide passes whose columns are split over workgroups (knob mfma_split = 1 wherever the shape fits) against the staged
    kernel (0), bit for bit: tiles that overlap, slices of different lengths and without columns, passes of 32 rows and the
    rest. `gemv` picks by shape; a workspace of NULL is the plain call."""
    w, x = weights_bf16(R, C, seed=180).cuda(), acts_bf16(M, C, seed=181).cuda()
    L, y = card.lib, torch.empty(M, R, dtype=torch.bfloat16, device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    try:
        card.set_tuning("gemv_mfma_from", 5)  # the staged kernel's shapes whatever their size, small ragged ones too
        card.set_tuning("mfma_split", 0)
        want = card.gemv(w, x)
        assert L.btb_hip_gemv_bf16_floats(R, C, M) == 0
        card.set_tuning("mfma_split", 1)
        floats = L.btb_hip_gemv_bf16_floats(R, C, M)
        # (more than sixteen rows of x over long rows of a ragged matrix are the column-interleaved kernel's)
        assert (floats > 0) == (M <= 16 or R % 16 == 0 or C <= 4096)
        if floats:
            ws = torch.full((floats + 64,), float("nan"), device="cuda")
            assert L.btb_hip_gemv_bf16_ws(p(w), p(x), p(y), R, C, M, p(ws), None) == 0
            torch.cuda.synchronize()
            assert torch.equal(y.view(torch.int16), want.view(torch.int16))
            assert torch.isnan(ws[floats:]).all()
            assert L.btb_hip_gemv_bf16_ws(p(w), p(x), p(y), R, C, M, ctypes.c_void_p(ws.data_ptr() + 4), None) == -6
            assert L.btb_hip_gemv_bf16_ws(p(w), p(x), p(y.zero_()), R, C, M, None, None) == 0
            torch.cuda.synchronize()
            assert torch.equal(y.view(torch.int16), want.view(torch.int16))
        card.set_tuning("mfma_split", -1)
        assert torch.equal(card.gemv(w, x).view(torch.int16), want.view(torch.int16))
    finally:
        card.set_tuning("mfma_split", -1)
        card.set_tuning("gemv_mfma_from", -1)


@pytest.mark.parametrize("R,C,M,eager", [(1024, 3072, 16, False), (512, 3584, 32, False), (1536, 5120, 16, False), (1024, 7168, 12, True),
                                         (1536, 5120, 17, True), (2560, 9728, 32, True), (6144, 5120, 16, True)])
def test_an_eager_call_takes_a_second_launch_only_where_it_gains(card, monkeypatch, R, C, M, eager):
    """The columns split over workgroups take two launches and an allocation: a recorded call takes them wherever the library offers,
    an eager one where the kernels save more than the host pays; the bits are the same."""
    w, x, called = weights_bf16(R, C, seed=182).cuda(), acts_bf16(M, C, seed=183).cuda(), []
    assert card.lib.btb_hip_gemv_bf16_floats(R, C, M) > 0
    inner = type(card)._call
    monkeypatch.setattr(type(card), "_call", lambda self, name, *args: (called.append(name), inner(self, name, *args))[1])
    want, y = card.gemv(w, x), torch.empty(M, R, dtype=torch.bfloat16, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        card.gemv(w, x, y)
    assert called == ["btb_hip_gemv_bf16_ws" if eager else "btb_hip_gemv_bf16", "btb_hip_gemv_bf16_ws"]
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("R,C", [(16, 32), (17, 544), (4128, 512), (16416, 640), (48, 672), (12336, 1024), (1001, 1280),
                                 (6144, 1312), (32, 2048), (5003, 2080), (2560, 2560), (8224, 2528), (2560, 2592), (3008, 3136),
                                 (4096, 3584), (1536, 4096), (32, 4000)])
@pytest.mark.parametrize("M", [5, 8, 16, 17, 32, 40])
def test_two_tiles_of_weights_in_flight_change_no_bit(card, R, C, M):
    """The kernel with two tiles of weights in flight (knob mfma_ahead = 1: wherever the shape fits, 0: nowhere, -1: by the rule)
    against the staged one, bit for bit, plain and with the gate / up fold: one to many turns a workgroup, odd and even, tiles of
    10, 12 and 16 rows and overlapping ones, slices shorter than the kernel's and waves without a step, non-finite weights in rows
    of their own. From five rows on whatever the shape, so that the small ragged matrices reach both kernels."""
    w, x = weights_bf16(R, C, seed=190), acts_bf16(M, C, seed=191).cuda()
    w[R // 2, C - 1], w[R - 1, 0] = float("nan"), float("inf")
    w, got = w.cuda(), []
    try:
        card.set_tuning("gemv_mfma_from", 5)
        for knob in (0, 1, -1):
            card.set_tuning("mfma_ahead", knob)
            got.append([card.gemv(w, x)] + ([card.gemv_glu_silu(w, x)] if R % 32 == 0 else []))
    finally:
        card.set_tuning("mfma_ahead", -1)
        card.set_tuning("gemv_mfma_from", -1)
    for want, *others in zip(*got):
        for y in others:
            assert torch.equal(y.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("R,C", [(16, 72), (17, 520), (512, 536), (100, 648), (4097, 1016), (1001, 1288), (2560, 2056), (5003, 2552),
                                 (2560, 2568), (300, 3000), (9000, 3000), (1536, 3592), (33, 4088)])
@pytest.mark.parametrize("M", [5, 8, 16, 17, 33])
def test_rows_of_no_multiple_of_32_columns_on_the_matrix_cores(card, R, C, M):
    """Rows whose last step of 32 columns is short, against 64 bits: the output's rounding (bf16 has eight significant bits: half
    a step is at most 2^-8 of the value) and C roundings of 2^-24 of the sum of magnitudes, twice over for the accumulator's own;
    a non-finite weight at a row's end stays in its row, non-finite x in its own."""
    w, x = weights_bf16(R, C, seed=200), acts_bf16(M, C, seed=201)
    w[1, C - 1], w[3, C - 8], w[R - 1, 0] = float("nan"), float("inf"), float("-inf")
    x[M - 1, C - 1] = float("nan")
    y = card.gemv(w.cuda(), x.cuda()).float().cpu().double()
    ref = x.double() @ w.double().T
    assert bool(y[: M - 1, 1].isnan().all()) and bool(y[M - 1].isnan().all())
    assert not bool(y[: M - 1, [r for r in (3, R - 1) if r != 1]].isfinite().any())
    keep = [r for r in range(R) if r not in (1, 3, R - 1)]
    y, ref = y[: M - 1, keep], ref[: M - 1, keep]
    bound = 2.0**-8 * ref.abs() * 1.01 + 2 * C * 2.0**-24 * (x[: M - 1].double().abs() @ w[keep].double().abs().T)
    assert bool(((y - ref).abs() <= bound).all())


@pytest.mark.parametrize("R,C,M", [(16, 72, 5), (34, 520, 8), (512, 648, 17), (1008, 1016, 33), (130, 1288, 6), (2576, 2056, 12),
                                   (5006, 2552, 16), (2560, 2568, 20), (300, 3000, 5), (1536, 3592, 16), (16, 4088, 8)])
def test_the_forms_of_rows_of_no_multiple_of_32_columns_agree(card, R, C, M):
    """From five rows of x on, over rows whose last step of 32 columns is short: the gate / up fold has the bits of the matvec and
    silu_mul, the add + norm forms those of add_rmsnorm and the matvec, a row those it has in a narrower pass."""
    bits = lambda t: t.view(torch.int16)
    empty = lambda rows, cols: torch.empty(rows, cols, dtype=torch.bfloat16, device="cuda")
    w, x, d = weights_bf16(R, C, seed=210).cuda(), acts_bf16(M, C, seed=211).cuda(), acts_bf16(M, C, seed=212).cuda()
    nw = (1.0 + 0.1 * torch.randn(C, generator=torch.Generator().manual_seed(213))).to(torch.bfloat16).cuda()
    y = card.gemv(w, x)
    m = empty(M, R // 2)
    card.silu_mul(y, m)
    assert torch.equal(bits(card.gemv_glu_silu(w, x)), bits(m))
    assert torch.equal(bits(card.gemv(w, x[:5].contiguous())), bits(y[:5]))
    for add in (d, None):
        h, xn, h2 = x.clone(), empty(M, C), empty(M, C)
        card.add_rmsnorm(h, add, nw, 1e-6, xn)
        want = card.gemv(w, xn)
        got = card.gemv_norm(w, x, add, nw, 1e-6, h2, empty(M, R))
        assert torch.equal(bits(got), bits(want)) and torch.equal(bits(h2), bits(h))
        card.silu_mul(want, m)
        got = card.gemv_norm(w, x, add, nw, 1e-6, h2.zero_(), empty(M, R // 2), glu=True)
        assert torch.equal(bits(got), bits(m)) and torch.equal(bits(h2), bits(h))
        got = card.gemv_norm(w, x, add, nw, 1e-6, None, empty(M, R), centered=True)
        card.add_rmsnorm(x.clone(), add, nw, 1e-6, xn, centered=True)
        assert torch.equal(bits(got), bits(card.gemv(w, xn)))
    ids = torch.arange(M - 1, -1, -1, dtype=torch.int32, device="cuda")
    card.add_rmsnorm(x.flip(0).contiguous(), None, nw, 1e-6, xn)
    got = card.gemv_embed_norm(w, x, ids, nw, 1e-6, h2, empty(M, R))
    assert torch.equal(bits(got), bits(card.gemv(w, xn))) and torch.equal(bits(h2), bits(x.flip(0)))


@pytest.mark.parametrize("R,C,M", [(34, 520, 8), (1008, 1016, 33), (2576, 2056, 12), (300, 3000, 5)])
def test_knobs_over_rows_of_no_multiple_of_32_columns(card, R, C, M):
    """The knobs that choose a kernel within the matrix-core family move no bit of such rows, `gemv_no_mfma` and `gemv_mfma_from`
    choose the family as they do for other rows."""
    bits = lambda t: t.view(torch.int16)
    w, x = weights_bf16(R, C, seed=214).cuda(), acts_bf16(M, C, seed=215).cuda()
    y = card.gemv(w, x)
    try:
        for knob in ("mfma_ahead", "mfma_lds", "mfma_tile_rows"):
            card.set_tuning(knob, 0)
            assert torch.equal(bits(card.gemv(w, x)), bits(y)), knob
            card.set_tuning(knob, -1)
        card.set_tuning("gemv_no_mfma", 1)
        vector = card.gemv(w, x)
        card.set_tuning("gemv_no_mfma", -1)
        card.set_tuning("gemv_mfma_from", M + 1)
        assert torch.equal(bits(card.gemv(w, x)), bits(vector))
        card.set_tuning("gemv_mfma_from", 2)
        assert torch.equal(bits(card.gemv(w, x[:3].contiguous())), bits(y[:3]))
    finally:
        for knob in ("mfma_ahead", "mfma_lds", "mfma_tile_rows", "gemv_no_mfma", "gemv_mfma_from"):
            card.set_tuning(knob, -1)
