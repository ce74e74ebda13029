"""Gathered contexts packed in sequence order: bit-exact against plain indexing of the cache."""

from __future__ import annotations

import pytest
import torch

from wavelet_amd import PagedKVCache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 2, 64, 65, 1024, 1025])
@pytest.mark.parametrize("kv_dtype,dequant", [("bf16", False), ("fp8_e4m3", False), ("fp8_e4m3", True)])
def test_gather_starts_every_sequence_after_those_before_it(cuda, batch, kv_dtype, dequant):
    """Up to 1,024 sequences a workgroup adds up the lengths before its own, past that a prefix sum is handed in:
    empty sequences first, last and in between, a wave's worth of lengths and one more; the total given or not."""
    h, d, bs = 2, 64, 16
    gen = torch.Generator().manual_seed(batch)
    lens = torch.randint(0, 40, (batch,), generator=gen)
    lens[torch.rand(batch, generator=gen) < 0.2] = 0
    lens[0], lens[-1] = (0, 0) if batch > 2 else (33, 17)
    nb = 3 * batch
    table = torch.randperm(nb, generator=gen)[:3 * batch].view(batch, 3).to(torch.int32)
    cache = PagedKVCache(nb, bs, h, d, kv_dtype=kv_dtype, device=cuda)
    for t in (cache.k, cache.v):
        t.view(torch.uint8).copy_(torch.randint(0, 0x7F, t.view(torch.uint8).shape, generator=gen, dtype=torch.uint8))
    if kv_dtype != "bf16":
        for t in (cache.k_scale, cache.v_scale):
            t.copy_(2.0 ** torch.randint(-6, 3, t.shape, generator=gen).float())
    k, v = cache.k.cpu(), cache.v.cpu()
    if dequant:
        k, v = (x.view(torch.float8_e4m3fn).float() for x in (k, v))
        k = (k * cache.k_scale.cpu()[:, :, None, None, None]).to(torch.bfloat16)
        v = (v * cache.v_scale.cpu()[:, :, None, None]).to(torch.bfloat16)
    k = k.permute(0, 3, 1, 2, 4).reshape(nb, bs, h, d)  # [block, token, head, d]
    v = v.permute(0, 3, 1, 2)
    want = [torch.cat([x[table[i].long()].flatten(0, 1)[:n] for i, n in enumerate(lens.tolist())]) for x in (k, v)]
    for total in (None, int(lens.sum())):
        got = cache.gather(table.to(cuda), lens.to(torch.int32).to(cuda), dequant=dequant, total_tokens=total)
        for g, w in zip(got, want):
            assert torch.equal(g.cpu().view(torch.uint8), w.contiguous().view(torch.uint8))
