"""Decode at the edges of the launch shapes the library chooses by size, against the oracle."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch
from kvcase import bits_of, check_attention, to_dev_bits
from oracle import paged
from wavelet_amd import PagedKVCache, _lib, decode_plan, paged_decode_gqa, synth

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.mark.parametrize("bs", [16, 32, 64])
@pytest.mark.parametrize("top", [512, 513, 700, 896, 897, 1023])
@pytest.mark.parametrize("hq,hkv,d", [(14, 2, 64), (32, 8, 128)])
def test_contexts_around_the_single_workgroup_range(cuda, hq, hkv, d, top, bs):
    """Narrow rows of 5 to 7 partitions: the longest context at both ends of the range and past them, with contexts of one token, of
    less than a wave's share and none at all beside it; the same step with the partition given
    (two workgroups and a merge) agrees. d=128 bf16 keeps the two."""
    lens = np.array([top, 1, 0, 15, top // 8, top // 8 + 1, 511, top - 1])
    _check(cuda, hq, hkv, d, bs, lens)


@pytest.mark.parametrize("hq,hkv,d,bs,lens", [
    (32, 8, 128, 16, [1024]),  # one workgroup per sequence and head
    (32, 8, 128, 16, [1025]),  # spread: partitions of 64, four waves
    (32, 8, 128, 64, [2048, 1, 257, 0]),
    (32, 8, 128, 16, [2049, 513, 16]),  # spread: partitions of 128
    (14, 2, 64, 32, [1999, 2048, 255, 1024, 1025]),
    (14, 2, 64, 16, [4096, 33]),  # eight slots, narrow
    (14, 2, 64, 16, [4097, 2048]),  # nine: not spread
    (32, 8, 128, 128, [1500, 300]),
    (28, 4, 128, 16, [8192] * 4 + [700]),  # 5 x 4 heads x 16 slots: more than one per CU
])
def test_few_long_contexts_spread_over_the_chip(cuda, hq, hkv, d, bs, lens):
    """Both sides of each bound of the rule that spreads few long contexts over more, smaller
    workgroups; the given partition agrees."""
    _check(cuda, hq, hkv, d, bs, np.array(lens))


def _check(cuda, hq, hkv, d, bs, lens):
    top = int(lens.max())
    w = synth.make_decode_workload(f"shape{d}t{top}b{bs}", batch=len(lens), num_kv_heads=hkv, num_q_heads=hq,
                                   head_dim=d, block_size=bs, context_lens=lens)
    gen = np.random.default_rng(top)
    kc, vc = paged.empty_cache(w.num_blocks, bs, hkv, d)
    kc[...] = paged.f32_to_bf16(gen.standard_normal(kc.shape).astype(np.float32))
    vc[...] = paged.f32_to_bf16(gen.standard_normal(vc.shape).astype(np.float32))
    q = synth.normal_bf16(synth.stream_key(w.name, "q"), (w.batch, hq, d))
    cache = PagedKVCache(w.num_blocks, bs, hkv, d, device=cuda)
    cache.k.copy_(to_dev_bits(kc, BF16, cuda).view(cache.k.shape))
    cache.v.copy_(to_dev_bits(vc, BF16, cuda).view(cache.v.shape))
    args = (to_dev_bits(q, BF16, cuda), cache, torch.from_numpy(w.block_tables).to(cuda),
            torch.from_numpy(w.context_lens).to(cuda), w.scale)
    kl, vl = paged.logical_kv(kc, vc)
    ref = paged.decode_gqa(paged.bf16_to_f32(q), paged.bf16_to_f32(kl), paged.bf16_to_f32(vl), w.block_tables,
                           w.context_lens, w.scale)
    for p in (0, 128):
        got = paged.bf16_to_f32(bits_of(paged_decode_gqa(*args, partition_size=p)))
        check_attention(got, ref, f"{w.name} P={p}")
    return w, args, ref


@pytest.mark.parametrize("hq,hkv,d,lens", [(32, 8, 128, [4000]), (32, 8, 128, [2048, 1500]), (14, 2, 64, [2048, 33])])
def test_a_workspace_of_the_planned_shape_is_enough(cuda, hq, hkv, d, lens):
    """A caller that sized its workspace by decode_plan's shape (half the slots the launch would take
    with more) is served with it, and one byte less is refused."""
    w, (q, cache, bt, sl, scale), ref = _check(cuda, hq, hkv, d, 16, np.array(lens))
    lib = _lib.load()
    top = max(lens)
    part, waves, chunks = decode_plan(w.batch, hkv, top, 16)
    need = lib.wkv_decode_workspace_size(w.batch, hq, d, top, part * waves)
    assert chunks > 1 and need < lib.wkv_decode_workspace_size(w.batch, hq, d, top, 0)
    ws = torch.empty(need, dtype=torch.uint8, device=cuda)
    out = torch.full((w.batch, hq, d), float("nan"), dtype=BF16, device=cuda)
    args = (ctypes.byref(cache.descriptor()), q.data_ptr(), q.stride(0), q.stride(1), out.data_ptr(), hq, bt.data_ptr(),
            bt.stride(0), bt.shape[1], sl.data_ptr(), w.batch, top, ctypes.c_float(scale), 0, ws.data_ptr())
    stream = torch.cuda.current_stream(cuda).cuda_stream
    assert lib.wkv_paged_decode_gqa(*args, need - 1, None, stream) == _lib.WKV_ERR_INVALID
    _lib.check(lib.wkv_paged_decode_gqa(*args, need, None, stream), "planned workspace")
    check_attention(paged.bf16_to_f32(bits_of(out)), ref, w.name)
