"""The decode step's products (csrc/skinny_linear.hip) against float64, and their fused forms
against the separate kernels bit for bit.

Bound of a product: fp32 sums of K exact bf16 products in any order are within K 2^-24 sum|x w| of
the exact sum, and the bf16 result within half a spacing (2^-8 relative, safely) of that.  It is the worst
case, far above the errors of a correct sum: test_exact_sums holds them to none.
"""

from __future__ import annotations

import pytest
import torch

from int8kv import decode_loop as DL

pytestmark = pytest.mark.gpu

# One block of K; slots of unequal length (24 blocks on 8 waves, 41 on 8); eight full slots; K split
# over groups of workgroups (65 blocks, and the 18944-wide down projection's 296); row blocks
# below, at and above one per compute unit.
SHAPES = [(64, 16), (512, 2048), (1536, 48), (2624, 4112), (4096, 4096), (4160, 64), (18944, 3584)]


def _inputs(rows, k, n, dev, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn(rows, k, generator=g, device=dev).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g, device=dev) * 0.05).to(torch.bfloat16)
    b = torch.randn(n, generator=g, device=dev).to(torch.bfloat16)
    work = torch.empty(max(DL.linear_workspace_bytes(rows, w), 16), dtype=torch.uint8, device=dev)
    return x, w, b, work


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 32])
@pytest.mark.parametrize("k,n", SHAPES)
def test_linear_matches_float64(cuda, rows, k, n):
    x, w, b, work = _inputs(rows, k, n, cuda, rows + k)
    out = torch.full((rows + 1, n), float("nan"), dtype=torch.bfloat16, device=cuda)
    for bias in (None, b):
        DL.hip_linear(x, w, bias, out[:rows], work)
        ref = x.double() @ w.double().t() + (0 if bias is None else bias.double())
        mass = x.double().abs() @ w.double().abs().t()
        err = (out[:rows].double() - ref).abs()
        assert (err <= 2.0**-8 * ref.abs() + k * 2.0**-24 * (mass + ref.abs())).all()
        assert torch.isnan(out[rows]).all(), "a row past x was written"


@pytest.mark.parametrize("rows", [1, 17, 32])
@pytest.mark.parametrize("k,n", [(64, 16), (2624, 48), (4096, 64), (4160, 64), (18944, 3584), (32768, 32)])
def test_exact_sums(cuda, rows, k, n):
    """Whole numbers whose products and sums fp32 holds exactly (at most 8 x 4 x K < 2^24): the
    result is the exact sum rounded to bf16, whatever the order; a column of K left out or a partial sum
    kept in fewer bits changes it.  The fused residual add sums the same way."""
    g = torch.Generator(device=cuda).manual_seed(rows + k)
    x = torch.randint(-8, 9, (rows, k), generator=g, device=cuda).to(torch.bfloat16)
    w = torch.randint(-4, 5, (n, k), generator=g, device=cuda).to(torch.bfloat16)
    b = torch.randint(-64, 65, (n,), generator=g, device=cuda).to(torch.bfloat16)
    work = torch.empty(max(DL.linear_workspace_bytes(rows, w), 16), dtype=torch.uint8, device=cuda)
    out = torch.empty(rows, n, dtype=torch.bfloat16, device=cuda)
    exact = x.double() @ w.double().t()
    assert torch.equal(DL.hip_linear(x, w, b, out, work), (exact + b.double()).to(torch.bfloat16))
    residual = torch.randint(-100, 101, (rows, n), generator=g, device=cuda).to(torch.bfloat16)
    want = (residual.double() + exact.to(torch.bfloat16).double()).to(torch.bfloat16)
    DL.hip_linear_add_rms_norm(x, w, residual, torch.ones_like(b), torch.empty_like(out), 1e-6, work)
    assert torch.equal(residual, want)


@pytest.mark.parametrize("rows", [1, 16, 32])
@pytest.mark.parametrize("k,ffn", [(64, 8), (512, 1024), (3584, 2376)])
def test_linear_silu_mul_equals_the_two_kernels(cuda, rows, k, ffn):
    x, w, _, work = _inputs(rows, k, 2 * ffn, cuda, 7 * rows + k)
    gate_up = torch.empty(rows, 2 * ffn, dtype=torch.bfloat16, device=cuda)
    ref = torch.empty(rows, ffn, dtype=torch.bfloat16, device=cuda)
    out = torch.empty_like(ref)
    DL.hip_silu_mul(DL.hip_linear(x, w, None, gate_up, work), ref)
    DL.hip_linear_silu_mul(x, w, out)
    assert torch.equal(out, ref)


@pytest.mark.parametrize("rows", [1, 16, 32])
@pytest.mark.parametrize("k,n", [(512, 512), (3584, 3584), (4160, 64), (18944, 3584), (64, 8192)])
def test_linear_add_rms_norm_equals_the_two_kernels(cuda, rows, k, n):
    x, w, b, work = _inputs(rows, k, n, cuda, 11 * rows + k)
    residual = torch.randn(rows, n, device=cuda).to(torch.bfloat16)
    ref_res, ref = residual.clone(), torch.empty_like(residual)
    DL.hip_add_rms_norm(ref_res, DL.hip_linear(x, w, None, torch.empty_like(residual), work), b, ref, 1e-6)
    out = torch.empty_like(residual)
    DL.hip_linear_add_rms_norm(x, w, residual, b, out, 1e-6, work)
    assert torch.equal(residual, ref_res)
    # The row's sum of squares is added in another order: at most one bf16 step of each rounding.
    assert ((out.double() - ref.double()).abs() <= 2.0**-6 * ref.double().abs()).all()


def test_non_finite_values_stay_in_their_rows_and_columns(cuda):
    x, w, _, work = _inputs(20, 512, 64, cuda, 3)
    x[3, 100] = float("nan")
    w[5, 7] = float("inf")
    out = DL.hip_linear(x, w, None, torch.empty(20, 64, dtype=torch.bfloat16, device=cuda), work)
    ref = x.double() @ w.double().t()
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    assert torch.equal(torch.isposinf(out), torch.isposinf(ref))
    assert torch.equal(torch.isneginf(out), torch.isneginf(ref))


def test_what_the_kernels_take(cuda):
    w = torch.zeros(64, 128, dtype=torch.bfloat16, device=cuda)
    assert DL.skinny_linear_ok(1, w) and DL.skinny_linear_ok(32, w)
    assert not DL.skinny_linear_ok(33, w) and not DL.skinny_linear_ok(0, w)
    assert not DL.skinny_linear_ok(1, w[:, :96]) and not DL.skinny_linear_ok(1, w[:24])
    assert not DL.skinny_linear_ok(1, w[:, 4:68]) and not DL.skinny_linear_ok(1, w.float())


@pytest.mark.parametrize("batch,hidden", [(33, 512), (3, 480)])
def test_step_falls_back_to_torch_products(cuda, batch, hidden):
    shape = DL.QwenShape(hidden=hidden, layers=1, q_heads=28, kv_heads=4, head_dim=128, ffn=1024, vocab=2048)
    weights = DL.random_weights(shape, cuda, seed=1)
    loop = DL.DecodeLoop(weights, batch, 5, 2, "bf16")
    assert loop.partials is None
    loop.prefill(torch.zeros(batch, 5, dtype=torch.int64))
    loop.step_eager()
    assert torch.isfinite(loop.logits.float()).all()


def test_silu_of_every_bf16_value(cuda):
    """All 65536 gate values (both branches of silu.h, infinities, NaN, denormals) and the fused
    product's copy of it: within half a bf16 spacing, with 2^-10 of one for the fp32 error, of the
    float64 value; -0 where exp(-g) overflows fp32; a NaN stays one and -inf becomes one, as in
    torch.nn.functional.silu."""
    bits = torch.arange(1 << 16, dtype=torch.int32)
    gate = (bits << 16).view(torch.float32).to(torch.bfloat16).view(32, 2048)
    ref = gate.double() / (1 + torch.exp(-gate.double()))
    overflows = (gate.double() < -88.7228394) & torch.isfinite(gate)
    ref = torch.where(overflows, torch.zeros_like(ref), ref)
    assert torch.equal(torch.isnan(ref), torch.isnan(torch.nn.functional.silu(gate.double())))
    gate_up = torch.cat([gate, torch.ones_like(gate)], dim=1).to(cuda)
    out = DL.hip_silu_mul(gate_up, torch.empty(32, 2048, dtype=torch.bfloat16, device=cuda)).cpu().double()
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    fine = torch.isfinite(ref)
    assert torch.equal(out[torch.isinf(ref)], ref[torch.isinf(ref)])
    spacing = torch.exp2(torch.floor(torch.log2(ref[fine].abs().clamp_min(2.0**-126))) - 7)
    assert ((out[fine] - ref[fine]).abs() <= spacing * (0.5 + 2.0**-10)).all()
    # The fused product with w = a diagonal gives the same values (column 5 overflows to -inf in
    # row 3 and +inf in row 4: inputs of -inf itself would put 0 x inf into the other columns).
    x = torch.zeros(32, 64, dtype=torch.bfloat16, device=cuda)
    x[:, :16] = torch.randn(32, 16, device=cuda).to(torch.bfloat16) * 120
    x[3, 5], x[4, 5] = -3e38, 3e38
    diag = torch.ones(16, device=cuda)
    diag[5] = 2.0**40
    w = torch.zeros(32, 64, dtype=torch.bfloat16, device=cuda)
    w[:16, :16] = torch.diag(diag)
    w[16:, 0] = 1
    fused = DL.hip_linear_silu_mul(x, w, torch.empty(32, 16, dtype=torch.bfloat16, device=cuda))
    gate = (x[:, :16].float() * diag).to(torch.bfloat16)
    gu = torch.cat([gate, x[:, :1].expand(32, 16)], dim=1).contiguous()
    ref = DL.hip_silu_mul(gu, torch.empty_like(fused))
    assert torch.isnan(ref[3, 5]) and torch.isinf(ref[4, 5]) and torch.isnan(ref).sum() == 1
    assert torch.equal(torch.isnan(fused), torch.isnan(ref))
    assert torch.equal(torch.nan_to_num(fused), torch.nan_to_num(ref))
