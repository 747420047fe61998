"""Cache writes on both sides of the row kernels' bounds (one 16-byte load per lane: fp32 sources at
every size, 16-bit ones below 2^20 elements), bit-exact against the oracle."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

import int8kv
from int8kv import _lib, cache_ops
from oracle import int8kv_oracle as O

pytestmark = pytest.mark.gpu

# (tokens, kv heads, head_dim): one token; rows of 10 pieces; kv heads no power of two; more lanes
# per token than a wave; 2^20 elements and one token fewer; fp32 past the Infinity Cache
# (256 MB) and on both sides of half of it, odd token counts among them.
SHAPES = [(1, 4, 128), (37, 2, 80), (130, 3, 64), (63, 8, 256), (2047, 4, 128), (2048, 4, 128)]
LARGE = [(60000, 4, 128), (70000, 3, 128), (26215, 4, 128), (13107, 8, 128)]
DTYPES = [torch.float32, torch.bfloat16, torch.float16]


def _inputs(tokens, hkv, d, dtype, dev, seed):
    g = torch.Generator().manual_seed(seed)
    k = (torch.randn(tokens, hkv, d, generator=g) * 3).to(dtype)
    v = torch.randn(tokens, hkv, d, generator=g).to(dtype)
    blocks = tokens // 16 + 2
    slots = torch.randperm(blocks * 16, generator=g)[:tokens]
    slots[::7] = -1
    if tokens > 2:
        slots[1] = blocks * 16 + 5  # past the cache
    return k, v, slots, torch.zeros(blocks, 16, hkv, d, dtype=torch.int8)


@pytest.mark.parametrize("tokens,hkv,d,dtype", [(*s, t) for s in SHAPES for t in DTYPES]
                         + [(*s, torch.float32) for s in LARGE])
def test_static_write(cuda, tokens, hkv, d, dtype):
    k, v, slots, cache = _inputs(tokens, hkv, d, dtype, cuda, tokens + d)
    ks = torch.linspace(0.01, 0.08, hkv)
    vs = torch.linspace(0.03, 0.005, hkv)
    kc, vc = cache.to(cuda), cache.to(cuda)
    int8kv.int8_kv_cache_write(k.to(cuda), v.to(cuda), kc, vc, slots.to(cuda), ks.to(cuda), vs.to(cuda))
    rk, rv = cache.numpy().copy(), cache.numpy().copy()
    keep = (slots >= 0) & (slots < cache.shape[0] * 16)
    O.int8_kv_cache_write(k[keep].float().numpy(), v[keep].float().numpy(), rk, rv,
                          slots[keep].numpy(), ks.numpy(), vs.numpy())
    assert np.array_equal(kc.cpu().numpy(), rk) and np.array_equal(vc.cpu().numpy(), rv)


@pytest.mark.parametrize("strided_scales", [False, True])
@pytest.mark.parametrize("tokens,hkv,d,dtype", [
    (*s, t) for s in [s for s in SHAPES if s[2] != 80] + [(40, 4, 512), (40, 4, 256)] for t in DTYPES[:2]]
    + [(*s, torch.float32) for s in LARGE])
def test_dynamic_write(cuda, tokens, hkv, d, dtype, strided_scales):
    k, v, slots, cache = _inputs(tokens, hkv, d, dtype, cuda, 3 * tokens + d)
    kc, vc = cache.to(cuda), cache.to(cuda)
    step = 2 if strided_scales else 1
    ksc, vsc = (torch.zeros(cache.shape[0], 16, hkv * step, device=cuda)[..., ::step] for _ in range(2))
    cache_ops.reshape_and_cache_int8(k.to(cuda), v.to(cuda), kc, vc, ksc, vsc, slots.to(cuda))
    rk, rv = cache.numpy().copy(), cache.numpy().copy()
    rks, rvs = (np.zeros((cache.shape[0], 16, hkv), np.float32) for _ in range(2))
    keep = (slots >= 0) & (slots < cache.shape[0] * 16)
    O.reshape_and_cache_int8(k[keep].float().numpy(), v[keep].float().numpy(), rk, rv, rks, rvs,
                             slots[keep].numpy())
    assert np.array_equal(kc.cpu().numpy(), rk) and np.array_equal(vc.cpu().numpy(), rv)
    assert np.array_equal(ksc.cpu().numpy(), rks) and np.array_equal(vsc.cpu().numpy(), rvs)


@pytest.mark.parametrize("dynamic", [False, True])
def test_more_pieces_than_one_launch_counts(cuda, dynamic):
    """2^31 pieces of 16 bytes and some more (16.8 M fp32 tokens x 4 x 128): two launches, of which the
    few rows written lie at the start, on both sides of the bound and at the end.  Every token reads
    the same source row (token stride 0), all other slots are skipped."""
    hkv, d, blocks = 4, 128, 4
    first = 0x7FFFFF00 // (hkv * d // 4)  # tokens of the first launch
    tokens = first + 1000
    g = torch.Generator().manual_seed(6)
    k, v = (torch.randn(1, hkv, d, generator=g) * 2 for _ in range(2))
    slots = torch.full((tokens,), -1, dtype=torch.int32, device=cuda)
    for i, t in enumerate((0, 5, first - 1, first, first + 1, tokens - 1)):
        slots[t] = 7 * i
    ks, vs = torch.full((hkv,), 0.03, device=cuda), torch.full((hkv,), 0.05, device=cuda)
    kc = torch.full((blocks, 16, hkv, d), 99, dtype=torch.int8, device=cuda)
    vc = kc.clone()
    ksc = torch.zeros(blocks, 16, hkv, device=cuda)
    vsc = ksc.clone()
    kd, vd, lib = k.to(cuda), v.to(cuda), _lib.load()
    src = (ctypes.c_int64 * 3)(0, d, 1)
    args = (kd.data_ptr(), vd.data_ptr(), _lib.F32, tokens, hkv, d, src, src, kc.data_ptr(), vc.data_ptr(),
            blocks, 16, _lib.strides(kc), _lib.strides(vc))
    tail = (slots.data_ptr(), _lib.I32)
    if dynamic:
        status = lib.int8kv_dynamic_cache_write(*args, ksc.data_ptr(), vsc.data_ptr(), _lib.strides(ksc),
                                                _lib.strides(vsc), *tail, _lib.stream_handle(cuda))
    else:
        status = lib.int8kv_cache_write(*args, *tail, ks.data_ptr(), vs.data_ptr(),
                                        _lib.stream_handle(cuda))
    _lib.check(status, "cache write")
    rk = np.full((blocks, 16, hkv, d), 99, np.int8)
    rv, rks, rvs = rk.copy(), np.zeros((blocks, 16, hkv), np.float32), np.zeros((blocks, 16, hkv), np.float32)
    where = np.arange(6) * 7
    ref_k, ref_v = k.expand(6, hkv, d).numpy(), v.expand(6, hkv, d).numpy()
    if dynamic:
        O.reshape_and_cache_int8(ref_k, ref_v, rk, rv, rks, rvs, where)
    else:
        O.int8_kv_cache_write(ref_k, ref_v, rk, rv, where, ks.cpu().numpy(), vs.cpu().numpy())
    assert np.array_equal(kc.cpu().numpy(), rk) and np.array_equal(vc.cpu().numpy(), rv)
    assert np.array_equal(ksc.cpu().numpy(), rks) and np.array_equal(vsc.cpu().numpy(), rvs)
