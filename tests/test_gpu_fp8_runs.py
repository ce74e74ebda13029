"""fp8 appends of runs in pieces of 16 tokens: codes and scales bit-exact against the oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch
from kvcase import to_dev_bits
from oracle import paged
from wavelet_amd import PagedKVCache, synth

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.mark.parametrize("d,bs,short", [(64, 16, True), (128, 16, True), (128, 64, True), (64, 64, False),
                                        (128, 16, False), (128, 32, False)])
def test_runs_match_oracle(cuda, d, bs, short):
    """Runs of 1, 15, 16, 17, 33, ... tokens (whole pieces, remainders, several pieces), starting
    at offset 0 and inside a block, over earlier codes that hold every e4m3 pattern (NaN codes and
    both zeros among them) under scales that grow and scales that do not, tokens in reverse slot
    order, NaN and infinities in some rows; calls below and above 64 tokens (both launch shapes)."""
    _check(cuda, d, bs, short, 64)


@pytest.mark.parametrize("d,bs", [(64, 16), (128, 16), (128, 64)])
def test_runs_of_a_prompt_sized_call_match_oracle(cuda, d, bs):
    """The same runs in one call of 4,096 tokens (skipped slots make up the number): the prompt launch."""
    _check(cuda, d, bs, False, 4096)


def _check(cuda, d, bs, short, pad):
    nb, h = 64, 2
    rng = np.random.default_rng(d + bs + short)
    kc, vc = paged.empty_cache(nb, bs, h, d, dtype=np.uint8, fill=0)
    kc[...] = rng.integers(0, 256, kc.shape)
    vc[...] = rng.integers(0, 256, vc.shape)
    ks = (2.0 ** rng.integers(-12, 2, (nb, h))).astype(np.float32)
    vs = (2.0 ** rng.integers(-12, 2, (nb, h))).astype(np.float32)
    cache = PagedKVCache(nb, bs, h, d, kv_dtype="fp8_e4m3", device=cuda)
    for dst, src in ((cache.k, kc), (cache.v, vc), (cache.k_scale, ks), (cache.v_scale, vs)):
        dst.copy_(torch.from_numpy(src).view(dst.shape))
    sizes = [n for n in (1, 2, 5, 15, 16, 17, 31, 33, 64) if n <= bs]
    blocks = iter(rng.permutation(nb))
    calls = []
    for n in sizes:
        for first in sorted({0, 1, bs - n}):
            if first + n <= bs:
                calls.append(next(blocks) * bs + first + np.arange(n))
    calls.append(next(blocks) * bs + np.arange(bs)[::-1])
    if not short:
        calls = [np.concatenate(calls + [np.full(pad, -1)])]
    for i, slots in enumerate(calls):
        slots = slots.astype(np.int64)
        assert (len(slots) >= 64) == (not short) or len(slots) == 64
        key, val = (synth.normal_bf16(synth.stream_key("fp8runs", d, bs, i, w), (len(slots), h, d), std=2.0)
                    for w in "kv")
        if i % 2 or not short:
            key.reshape(-1)[rng.integers(0, key.size, 3)] = (0x7FC0, 0xFFC0, 0x7F80)
            val.reshape(-1)[rng.integers(0, val.size, 2)] = (0xFFC1, 0x8000)
        paged.append_fp8(kc, vc, ks, vs, key, val, slots)
        cache.append(to_dev_bits(key, BF16, cuda), to_dev_bits(val, BF16, cuda), torch.from_numpy(slots).to(cuda))
        torch.cuda.synchronize()
        for name, got, want in (("k", cache.k, kc), ("v", cache.v, vc), ("k_scale", cache.k_scale, ks),
                                ("v_scale", cache.v_scale, vs)):
            assert np.array_equal(got.cpu().numpy().reshape(want.shape), want), f"call {i}: {name} differs"
