"""Decode over 5 to 7 chosen partitions of narrow rows: one workgroup of eight waves, against the oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch
from kvcase import bits_of, check_attention, to_dev_bits
from oracle import paged
from wavelet_amd import PagedKVCache, paged_decode_gqa, synth

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.mark.parametrize("bs", [16, 32, 64])
@pytest.mark.parametrize("top", [512, 513, 700, 896, 897, 1023])
@pytest.mark.parametrize("hq,hkv,d", [(14, 2, 64), (32, 8, 128)])
def test_contexts_around_the_single_workgroup_range(cuda, hq, hkv, d, top, bs):
    """The longest context at both ends of the range and past them, with contexts of one token, of
    less than a wave's share and none at all beside it; the same step with the partition given
    (two workgroups and a merge) agrees. d=128 bf16 keeps the two."""
    lens = np.array([top, 1, 0, 15, top // 8, top // 8 + 1, 511, top - 1])
    w = synth.make_decode_workload(f"narrow{d}t{top}b{bs}", batch=len(lens), num_kv_heads=hkv, num_q_heads=hq,
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
