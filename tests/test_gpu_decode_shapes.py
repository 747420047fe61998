"""Head sizes between 64, 128 and 256 and GQA groups above 16 on the decode kernels, against the
fp32 oracle.

The reference's kernels take any head_dim (src/triton_ops/int8_paged_attention.py:112-129 pads it
to a power of two under a mask) and any group (the grid there is one program per query head).
This build runs head_dim 64, 128 and 256 on their own kernels; a head_dim in between (a multiple
of 16: 80 for Phi-2, 96 for Phi-3-mini, 112, 160, 192, ...) runs the next one with the elements
past head_dim read from inside the row but meeting zero query elements, and its output columns
past head_dim never stored.  A group above 16 (multi-query attention: Falcon-7B's 71 query heads
on one kv head, 64 query heads per kv head, group 24 ...) takes one wave or workgroup per 16 query
heads of a kv head.

Every case checks the oracle bar, that empty sequences give zero rows, and -- through an output
view whose rows are wider than head_dim, filled with NaN -- that nothing past head_dim is written.
Layouts: automatic (ranges, per-sequence, split), forced range counts with both merge grids,
forced splits; INT8 and BF16 caches, fp32 queries, quantize_q, and the write-then-decode path.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import int8kv
from test_decode_plan import _columns as plan_columns
from cases import bf16_caches, decode_case, oracle_int8, ranges_call, to_dev
from conftest import MAX_ABS, MIN_COS, metrics
from int8kv import _decode, _lib
from oracle import int8kv_oracle as O

pytestmark = pytest.mark.gpu

LENS = [0, 1, 17, 31, 32, 33, 255, 256, 257, 1000, 4097, 2200]


def _check(out, ref, what):
    got = out.float().cpu().numpy()
    assert np.isfinite(got).all(), f"{what}: non-finite output"
    err, cos, _ = metrics(got, ref)
    print(f"{what}: max|diff|={err:.3e} cos={cos:.7f}", flush=True)
    assert err <= MAX_ABS and cos >= MIN_COS, f"{what}: max|diff|={err} cos={cos}"
    return err


def _wide_out(q):
    """An output view [B, Hq, D] inside NaN-filled rows of 256 elements: the columns past D must
    stay NaN."""
    B, Hq, D = q.shape
    full = torch.full((B, Hq, 256), float("nan"), dtype=q.dtype, device=q.device)
    return full, full[..., :D]


def _untouched(full, D, what):
    assert torch.isnan(full[..., D:]).all(), f"{what}: columns past head_dim were written"


def _decode_auto(q, kc, vc, bt, sl, ks, vs, flags=_lib.DECODE_ALL):
    full, out = _wide_out(q)
    _decode.paged_decode(q, kc, vc, bt, sl, ks, vs, out, 0, flags)
    torch.cuda.synchronize()
    return full, out


def _plan(q, kc, bt, num_ranges=0, flags=_lib.DECODE_ALL):
    B, Hq, D = q.shape
    nb, bs, hkv, _ = kc.shape
    return _lib.decode_plan(q.dtype, kc.dtype, B, Hq, hkv, D, nb, bs, bt.shape[1],
                            num_ranges=num_ranges, flags=flags)


@pytest.mark.parametrize("d", [80, 96, 112, 48, 160, 192])
def test_padded_head_dims_int8(cuda, d):
    hq, hkv = (32, 8) if d != 160 else (16, 4)
    c = decode_case(LENS, seed=d, hq=hq, hkv=hkv, head_dim=d, extra_blocks=7)
    t = to_dev(c, cuda)
    q, kc, vc, bt, sl, ks, vs = t
    ref = oracle_int8(c)
    full, out = _decode_auto(*t)
    print(f"d={d} auto plan: {_plan(q, kc, bt)['layout']}", flush=True)
    assert (out[0] == 0).all()
    _check(out, ref, f"int8 d={d} auto")
    _untouched(full, d, f"int8 d={d} auto")
    for splits in (1, 3):  # one range per sequence (by-range merge), three (by-sequence merge)
        full, out = _wide_out(q)
        ranges_call(t, cuda, splits=splits, out=out)
        _check(out, ref, f"int8 d={d} ranges x{splits}")
        _untouched(full, d, f"int8 d={d} ranges x{splits}")
    full, out = _wide_out(q)
    ranges_call(t, cuda, splits=None, out=out, min_tiles=2)
    _check(out, ref, f"int8 d={d} automatic ranges")
    for splits in (1, 4):  # per-sequence layout, split layout with 4 workgroups per sequence
        out = int8kv.int8_paged_attention(q, kc, vc, bt, sl, ks, vs, num_splits=splits)
        torch.cuda.synchronize()
        assert out.shape == (len(LENS), hq, d)
        _check(out, ref, f"int8 d={d} num_splits={splits}")
    out = int8kv.int8_paged_attention(q.float(), kc, vc, bt, sl, ks, vs)
    torch.cuda.synchronize()
    assert _check(out, ref, f"int8 d={d} fp32 query") <= 1e-3
    ref_q = O.paged_attention_ref(c.query.float().numpy(), c.kc, c.vc, c.block_tables.numpy(),
                                  c.seq_lens.numpy(), c.k_scale.numpy(), c.v_scale.numpy(),
                                  quantize_q=True)
    full, out = _wide_out(q)
    ranges_call(t, cuda, splits=2, quantize_q=True, out=out)
    _check(out, ref_q, f"int8 d={d} quantize_q")
    _untouched(full, d, f"int8 d={d} quantize_q")


@pytest.mark.parametrize("d", [80, 96, 192])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_padded_head_dims_16bit_cache(cuda, d, dtype):
    c = decode_case(LENS, seed=d + 1, hq=16, hkv=4, head_dim=d, extra_blocks=5)
    q = c.query.to(cuda)
    k_cpu, v_cpu = bf16_caches(c, dtype)
    ref = O.paged_attention_ref(c.query.float().numpy(), k_cpu.float().numpy(),
                                v_cpu.float().numpy(), c.block_tables.numpy(), c.seq_lens.numpy())
    k16, v16 = k_cpu.to(cuda), v_cpu.to(cuda)
    bt, sl = c.block_tables.to(cuda), c.seq_lens.to(cuda)
    full, out = _decode_auto(q, k16, v16, bt, sl, None, None)
    _check(out, ref, f"{dtype} d={d} auto")
    _untouched(full, d, f"{dtype} d={d} auto")
    for splits in (1, 4):
        out = int8kv.bf16_paged_attention(q, k16, v16, bt, sl, num_splits=splits)
        torch.cuda.synchronize()
        _check(out, ref, f"{dtype} d={d} num_splits={splits}")
    full, out = _wide_out(q)
    _decode.paged_decode(q, k16, v16, bt, sl, None, None, out, 3 * len(LENS))
    torch.cuda.synchronize()
    _check(out, ref, f"{dtype} d={d} ranges x3")
    _untouched(full, d, f"{dtype} d={d} ranges x3")


# (hq, hkv, head_dim): group 17 (two column tiles, the second one head), 24, 32 and 64 (MQA),
# Falcon-7B's 71 query heads on one kv head at head_dim 64, and a padded head_dim with group 20.
GROUPS = [(34, 2, 128), (48, 2, 128), (32, 1, 128), (64, 1, 128), (71, 1, 64), (40, 2, 96),
          (32, 1, 256)]


@pytest.mark.parametrize("hq,hkv,d", GROUPS)
def test_groups_above_16_int8(cuda, hq, hkv, d):
    c = decode_case(LENS, seed=hq + hkv, hq=hq, hkv=hkv, head_dim=d, extra_blocks=7)
    t = to_dev(c, cuda)
    q, kc, vc, bt, sl, ks, vs = t
    ref = oracle_int8(c)
    full, out = _decode_auto(*t)
    assert (out[0] == 0).all()
    _check(out, ref, f"int8 {hq}/{hkv} d={d} auto")
    _untouched(full, d, f"int8 {hq}/{hkv} d={d} auto")
    for splits in (1, 3):
        out = ranges_call(t, cuda, splits=splits)
        _check(out, ref, f"int8 {hq}/{hkv} d={d} ranges x{splits}")
    for splits in (1, 4):
        out = int8kv.int8_paged_attention(q, kc, vc, bt, sl, ks, vs, num_splits=splits)
        torch.cuda.synchronize()
        _check(out, ref, f"int8 {hq}/{hkv} d={d} num_splits={splits}")
    ref_q = O.paged_attention_ref(c.query.float().numpy(), c.kc, c.vc, c.block_tables.numpy(),
                                  c.seq_lens.numpy(), c.k_scale.numpy(), c.v_scale.numpy(),
                                  quantize_q=True)
    out = int8kv.int8_paged_attention(q, kc, vc, bt, sl, ks, vs, quantize_q=True)
    torch.cuda.synchronize()
    _check(out, ref_q, f"int8 {hq}/{hkv} d={d} quantize_q")


@pytest.mark.parametrize("hq,hkv,d", [(32, 1, 128), (71, 1, 64), (40, 2, 96)])
def test_groups_above_16_bf16_cache(cuda, hq, hkv, d):
    c = decode_case(LENS, seed=hq * 3 + hkv, hq=hq, hkv=hkv, head_dim=d, extra_blocks=5)
    q = c.query.to(cuda)
    k_cpu, v_cpu = bf16_caches(c)
    ref = O.paged_attention_ref(c.query.float().numpy(), k_cpu.float().numpy(),
                                v_cpu.float().numpy(), c.block_tables.numpy(), c.seq_lens.numpy())
    k16, v16 = k_cpu.to(cuda), v_cpu.to(cuda)
    bt, sl = c.block_tables.to(cuda), c.seq_lens.to(cuda)
    for splits in (None, 1, 4):
        out = int8kv.bf16_paged_attention(q, k16, v16, bt, sl, num_splits=splits)
        torch.cuda.synchronize()
        _check(out, ref, f"bf16 {hq}/{hkv} d={d} num_splits={splits}")


def test_short_and_long_batches_take_every_layout(cuda):
    """The automatic layouts at a padded head_dim with a group above 16: a short batch (per
    sequence), one long sequence (split) and a long batch (ranges), each against the oracle."""
    seen = set()
    for lens, seed in (([300, 12, 512, 0], 51), ([20000], 52), ([3000] * 24 + [0, 9000], 53)):
        c = decode_case(lens, seed=seed, hq=40, hkv=2, head_dim=80, extra_blocks=3)
        t = to_dev(c, cuda)
        q, kc, vc, bt = t[:4]
        seen.add(_plan(q, kc, bt)["layout"])
        full, out = _decode_auto(*t)
        _check(out, oracle_int8(c), f"lens={lens[:4]}... auto")
        _untouched(full, 80, "auto")
    assert seen == {"per_sequence", "split", "ranges"}, seen


def test_write_then_decode(cuda):
    """The cache-write kernel at head_dim 80 into a cache the padded decode reads."""
    lens = [700, 1, 0, 2500, 64]
    c = decode_case(lens, seed=61, hq=32, hkv=2, head_dim=80, extra_blocks=3)
    q, _, _, bt, sl, ks, vs = to_dev(c, cuda)
    kc = torch.zeros(c.kc.shape, dtype=torch.int8, device=cuda)
    vc = torch.zeros_like(kc)
    int8kv.int8_kv_cache_write(c.key.to(cuda), c.value.to(cuda), kc, vc, c.slots.to(cuda), ks, vs)
    torch.cuda.synchronize()
    written = c.slots.numpy()
    nb, bs = c.kc.shape[:2]
    flat = lambda x: x.reshape(nb * bs, *x.shape[2:])[written]
    assert np.array_equal(flat(kc.cpu().numpy()), flat(c.kc))
    assert np.array_equal(flat(vc.cpu().numpy()), flat(c.vc))
    out = int8kv.int8_paged_attention(q, kc, vc, bt, sl, ks, vs)
    torch.cuda.synchronize()
    _check(out, oracle_int8(c), "write then decode d=80")


# Groups above 16 with enough work for the kernel that holds several column tiles per wave: 2, 3,
# 4 and 5 tiles at head_dim 64, 2 and 3 at 128 (a last tile of one head; kv heads of two waves),
# padded head_dims, and sequences of 0 to 2 segments per range.
WIDE = [(17, 1, 64), (48, 1, 64), (64, 1, 64), (71, 1, 64), (96, 1, 64), (66, 2, 128), (48, 1, 128),
        (71, 1, 128), (40, 2, 96), (33, 1, 48)]
WIDE_LENS = [0, 1, 33, 9000, 255, 4097, 31, 64, 12345, 2200, 0, 700] + [1500] * 10


@pytest.mark.parametrize("cache", ["int8", "bf16", "fp16"])
@pytest.mark.parametrize("hq,hkv,d", WIDE)
def test_groups_above_16_several_tiles_per_wave(cuda, hq, hkv, d, cache):
    c = decode_case(WIDE_LENS, seed=hq * 5 + d, hq=hq, hkv=hkv, head_dim=d, extra_blocks=7)
    t = to_dev(c, cuda)
    q, kc, vc, bt, sl, ks, vs = t
    if cache == "int8":
        full, out = _decode_auto(*t)
        _check(out, oracle_int8(c), f"{hq}/{hkv} d={d} auto")
        _untouched(full, d, f"{hq}/{hkv} d={d} auto")
        out = ranges_call(t, cuda, splits=3)
        _check(out, oracle_int8(c), f"{hq}/{hkv} d={d} ranges x3")
        out = int8kv.int8_paged_attention(q.float(), kc, vc, bt, sl, ks, vs)
        assert _check(out, oracle_int8(c), f"{hq}/{hkv} d={d} fp32 query") <= 1e-3
        for query in (q, q.float()):  # quantised: the same integer scores from either dtype
            out = int8kv.int8_paged_attention(query, kc, vc, bt, sl, ks, vs, quantize_q=True)
            ref = O.paged_attention_ref(c.query.float().numpy(), c.kc, c.vc, c.block_tables.numpy(),
                                        c.seq_lens.numpy(), c.k_scale.numpy(), c.v_scale.numpy(),
                                        quantize_q=True)
            _check(out, ref, f"{hq}/{hkv} d={d} quantize_q")
        return
    k_cpu, v_cpu = bf16_caches(c, torch.bfloat16 if cache == "bf16" else torch.float16)
    ref = O.paged_attention_ref(c.query.float().numpy(), k_cpu.float().numpy(),
                                v_cpu.float().numpy(), c.block_tables.numpy(), c.seq_lens.numpy())
    out = int8kv.bf16_paged_attention(q, k_cpu.to(cuda), v_cpu.to(cuda), bt, sl)
    assert (out[0] == 0).all() and (out[10] == 0).all()
    _check(out, ref, f"{hq}/{hkv} d={d} {cache}")


# Column tiles spread over the waves of one kv head: 2 + 2 + 1, 3 + 2 and 5; 2 + 2 + 2 and 3 + 3;
# 2 + 2; 2 x 4 and 4 + 3; 2 + 1 and 3; a pair per kv head (query heads, kv heads, head_dim, batch, tokens,
# tiles per wave on 256 compute units).
@pytest.mark.parametrize("cache", ["int8", "bf16"])
@pytest.mark.parametrize("hq,hkv,d,batch,tokens,per_wave", [
    (71, 1, 64, 7, 2560, 2), (71, 1, 64, 9, 8192, 3), (71, 1, 64, 20, 8192, 5), (96, 1, 64, 6, 2560, 2),
    (96, 1, 64, 9, 8192, 3), (64, 1, 64, 9, 2560, 2), (112, 1, 48, 9, 2560, 2), (112, 1, 48, 13, 8192, 4),
    (48, 1, 128, 13, 4096, 2), (48, 1, 112, 13, 8192, 3), (50, 2, 64, 9, 2560, 2)])
def test_groups_above_16_spread_over_waves(cuda, hq, hkv, d, batch, tokens, per_wave, cache):
    columns = plan_columns(torch.int8 if cache == "int8" else torch.bfloat16, batch, hq, hkv, d,
                           tokens // 16)
    assert columns[0] == per_wave
    lens = [tokens] + [tokens - 37 * i for i in range(1, batch)]
    c = decode_case(lens, seed=hq + batch, hq=hq, hkv=hkv, head_dim=d, extra_blocks=5)
    q, kc, vc, bt, sl, ks, vs = to_dev(c, cuda)
    if cache == "int8":
        full, out = _decode_auto(q, kc, vc, bt, sl, ks, vs)
        _untouched(full, d, f"{hq}/{hkv} d={d} {batch}x{tokens}")
        ref = oracle_int8(c)
    else:
        k_cpu, v_cpu = bf16_caches(c)
        ref = O.paged_attention_ref(c.query.float().numpy(), k_cpu.float().numpy(),
                                    v_cpu.float().numpy(), c.block_tables.numpy(),
                                    c.seq_lens.numpy())
        out = int8kv.bf16_paged_attention(q, k_cpu.to(cuda), v_cpu.to(cuda), bt, sl)
    _check(out, ref, f"{cache} {hq}/{hkv} d={d} {batch}x{tokens}")


@pytest.mark.parametrize("cache", ["int8", "fp16"])
@pytest.mark.parametrize("hq,d,block", [(71, 64, 32), (71, 64, 256), (48, 128, 64), (40, 80, 16)])
def test_groups_above_16_views(cuda, hq, d, block, cache):
    """64-bit tables and lengths, tables, queries, caches and outputs that are views into wider
    tensors, blocks of other sizes, fp16 queries: column tiles shared by a wave as for plain tensors."""
    lens = [5000, 0, 700, 4097, 1, 2222, 4999, 31] + [3000 + 11 * i for i in range(12)]
    c = decode_case(lens, seed=hq + block, hq=hq, hkv=1, head_dim=d, block_size=block, extra_blocks=3)
    q, kc, vc, bt, sl, ks, vs = to_dev(c, cuda)
    assert plan_columns(torch.int8 if cache == "int8" else torch.float16, len(lens), hq, 1, d,
                        bt.shape[1], bs=block)[0] >= 2
    if cache == "fp16":
        k_cpu, v_cpu = bf16_caches(c, torch.float16)
        kc, vc = k_cpu.to(cuda), v_cpu.to(cuda)
        ref = O.paged_attention_ref(c.query.float().numpy(), k_cpu.float().numpy(),
                                    v_cpu.float().numpy(), c.block_tables.numpy(), c.seq_lens.numpy())
    else:
        ref = oracle_int8(c)
    kv = torch.stack([kc, vc], dim=1)  # [blocks, 2, block, 1, d]: K and V of a block side by side
    kc, vc = kv[:, 0], kv[:, 1]
    tables = torch.full((len(lens), 2 * bt.shape[1]), -5, dtype=torch.int64, device=cuda)
    tables[:, ::2] = bt
    query = torch.full((len(lens), hq + 2, d + 16), float("nan"), dtype=torch.float16, device=cuda)
    query[:, 1 : hq + 1, :d] = q.to(torch.float16)
    out = torch.full_like(query, 7.0)
    view = out[:, 1 : hq + 1, :d]
    _decode.paged_decode(query[:, 1 : hq + 1, :d], kc, vc, tables[:, ::2], sl.to(torch.int64),
                         ks if cache == "int8" else None, vs if cache == "int8" else None, view)
    torch.cuda.synchronize()
    _check(view, ref, f"{cache} {hq}/1 d={d} block {block}")
    view.fill_(7.0)
    assert (out == 7).all(), "written outside the output view"


@pytest.mark.parametrize("cache", ["int8", "bf16"])
def test_groups_above_16_non_finite_queries(cuda, cache):
    """A NaN, an infinity of either sign and a huge finite query row: the rows of those heads as one wave
    per tile gives them, all others untouched by them."""
    lens = [4096] * 20 + [17, 0]
    c = decode_case(lens, seed=77, hq=71, hkv=1, head_dim=64)
    q, kc, vc, bt, sl, ks, vs = to_dev(c, cuda)
    if cache == "bf16":
        kc, vc = (t.to(cuda) for t in bf16_caches(c))
        ks = vs = None
    plain = torch.empty_like(q)
    _decode.paged_decode(q, kc, vc, bt, sl, ks, vs, plain)
    bad = q.clone()
    bad[0, 3, 5], bad[1, 20, 1], bad[2, 70, 0], bad[3, 40] = float("nan"), float("inf"), float("-inf"), 3e38
    touched = torch.zeros(len(lens), 71, dtype=torch.bool, device=cuda)
    touched[0, 3] = touched[1, 20] = touched[2, 70] = touched[3, 40] = True
    out = torch.empty_like(q)
    _decode.paged_decode(bad, kc, vc, bt, sl, ks, vs, out)
    assert torch.equal(out[~touched], plain[~touched])
    # The same heads as groups of 16 or fewer: one wave per tile.
    for b, h in touched.nonzero().tolist():
        one = torch.empty(1, 1, 64, dtype=q.dtype, device=cuda)
        _decode.paged_decode(bad[b : b + 1, h : h + 1], kc, vc, bt[b : b + 1], sl[b : b + 1], ks, vs, one)
        assert torch.equal(torch.isnan(one[0, 0]), torch.isnan(out[b, h])), (b, h)
        same = one[0, 0] == out[b, h]
        near = (one[0, 0].float() - out[b, h].float()).abs() <= MAX_ABS
        assert (same | near | torch.isnan(one[0, 0])).all(), (b, h)


def test_groups_above_16_with_the_automatic_counts_workspace(cuda):
    """71 heads on one kv head at 64: a workspace of the automatic count's ranges (those of 5 kv
    heads), of any more, and one byte too few."""
    c = decode_case([4000 - 7 * i for i in range(40)], seed=5, hq=71, hkv=1, head_dim=64)
    q, kc, vc, bt, sl, ks, vs = to_dev(c, cuda)
    lib, ref = _lib.load(), oracle_int8(c)
    least = lib.int8kv_decode_workspace_bytes(71, 1, 64, 16, lib.int8kv_decode_auto_ranges(5))
    full = lib.int8kv_decode_workspace_bytes(71, 1, 64, 16, 0)
    assert full > least
    for given in (full, (full + least) // 2, least, least - 1):
        work = torch.full((full + 4096,), 0x5A, dtype=torch.uint8, device=cuda)
        out = torch.full_like(q, float("nan"))
        status = lib.int8kv_paged_decode(
            q.data_ptr(), _lib.DTYPE_CODE[q.dtype], 40, 71, 64, _lib.strides(q), kc.data_ptr(),
            vc.data_ptr(), _lib.I8, kc.shape[0], 16, 1, _lib.strides(kc), _lib.strides(vc), bt.data_ptr(),
            _lib.DTYPE_CODE[bt.dtype], bt.shape[1], _lib.strides(bt), sl.data_ptr(),
            _lib.DTYPE_CODE[sl.dtype], ks.data_ptr(), vs.data_ptr(), 64**-0.5, out.data_ptr(),
            _lib.strides(out), work.data_ptr(), given, 0, 0, _lib.DECODE_ALL, _lib.stream_handle(cuda))
        torch.cuda.synchronize()
        if given < least:
            with pytest.raises(_lib.Int8KVError, match="E_WORKSPACE"):
                _lib.check(status, "int8kv_paged_decode")
            assert torch.isnan(out).all()
            continue
        assert status == 0
        _check(out, ref, f"workspace {given}")
        assert (work[given:] == 0x5A).all(), "written past the workspace"


@pytest.mark.parametrize("cache", ["int8", "bf16"])
@pytest.mark.parametrize("hq,hkv,d", [(14, 2, 64), (28, 4, 128), (16, 8, 256)])
def test_one_tile_per_wave_bound(cuda, hq, hkv, d, cache):
    """Per-sequence workgroups at the bound of one tile per wave (8 waves, 4 at head_dim 256) and one
    block past it, single-pass and split: the instance with one tile in flight and the one with
    two, on sequences of no, one, some and all tiles."""
    waves = 8 if d <= 128 else 4
    for splits in (1, 4):
        most = splits * waves * 32
        for longest in (most, most + 16):
            lens = [longest, 0, 1, 31, 33, most // 2 + 5, most - 1, longest - 16]
            c = decode_case(lens, seed=longest + d, hq=hq, hkv=hkv, head_dim=d, extra_blocks=3)
            q, kc, vc, bt, sl, ks, vs = to_dev(c, cuda)
            if cache == "int8":
                ref = oracle_int8(c)
                out = int8kv.int8_paged_attention(q, kc, vc, bt, sl, ks, vs, num_splits=splits)
            else:
                k_cpu, v_cpu = bf16_caches(c)
                ref = O.paged_attention_ref(c.query.float().numpy(), k_cpu.float().numpy(),
                                            v_cpu.float().numpy(), c.block_tables.numpy(),
                                            c.seq_lens.numpy())
                out = int8kv.bf16_paged_attention(q, k_cpu.to(cuda), v_cpu.to(cuda), bt, sl,
                                                  num_splits=splits)
            assert (out[1] == 0).all()
            _check(out, ref, f"{cache} d={d} splits={splits} longest={longest}")
