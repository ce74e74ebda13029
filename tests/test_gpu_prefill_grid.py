"""Prefill launch grids: how query heads and tiles are packed into workgroups, by the sizes.
Against the float64 oracle."""

import pytest
import torch

from kvcase import to_dev_bits
from test_gpu_prefill import BF16, _case, _run_and_check
from test_gpu_prefill_shared import _shared_call
from wavelet_amd import prefill_gqa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv_dtype", ["bf16", "fp8_e4m3"])
@pytest.mark.parametrize("hq,hkv,d,qlens,ctx", [
    (14, 2, 64, [255, 64, 1, 33, 256, 200, 31, 100], 0),  # 256 groups of a tile's heads: a tile to itself
    (14, 2, 64, [257, 64, 1, 33, 256, 200, 31, 100], 0),  # 288: packed across tiles
    (16, 8, 128, [256, 1, 90, 17], 48),
    (16, 8, 128, [257, 1, 90, 17], 48),
    (5, 1, 128, [289, 0, 128, 7] * 4, 20),
])
def test_both_sides_of_the_packing_bounds(cuda, hq, hkv, d, qlens, ctx, kv_dtype):
    w, cache, host, new = _case(cuda, f"pfgrid{hq}{d}{max(qlens)}", hq, hkv, d, 16, qlens, [n + ctx + 1 for n in qlens],
                                kv_dtype)
    _run_and_check(cuda, w, cache, host, new, f"{hq}/{hkv} {max(qlens)}")


@pytest.mark.parametrize("kv_dtype", ["bf16", "fp8_e4m3"])
@pytest.mark.parametrize("hq,hkv,d,n_seq,shared", [(14, 2, 64, 8, 0), (16, 8, 128, 4, 0), (5, 1, 128, 16, 0),
                                                   (3, 3, 64, 1, 0), (14, 2, 64, 2, 24), (3, 1, 128, 2, 96),
                                                   (28, 4, 128, 2, 40)])
def test_values_of_later_tiles_that_are_not_finite(cuda, hq, hkv, d, n_seq, shared, kv_dtype):
    """Infinite and NaN values from token 160 on (a block's and a query tile's first) leave the 160 queries
    before them, in the same unit groups, and every other sequence as they are without them, bit for bit."""
    qlens = [270] * n_seq
    outs = []
    for poison in (False, True):
        w, cache, _, new = _case(cuda, f"pfnan{hq}{d}{n_seq}", hq, hkv, d, 16, qlens, [n + 48 for n in qlens], kv_dtype)
        kn, vn, q, nslots, cu = new
        if poison:
            vn = vn.copy()
            vn[160:270:2] = 0x7FC0
            vn[161:270:2] = 0x7FC0 if kv_dtype != "bf16" else 0xFF80
        new = (kn, vn, q, nslots, cu)
        if shared:
            outs.append(_shared_call(cuda, w, cache, new, shared)[0])
        else:
            outs.append(prefill_gqa(to_dev_bits(q, BF16, cuda), cache, torch.from_numpy(w.block_tables).to(cuda),
                                    torch.from_numpy(w.context_lens).to(cuda), torch.from_numpy(cu).to(cuda), w.scale,
                                    key=to_dev_bits(kn, BF16, cuda), value=to_dev_bits(vn, BF16, cuda),
                                    slot_mapping=torch.from_numpy(nslots).to(cuda)))
    clean, got = outs
    assert torch.isfinite(clean).all() and torch.isnan(got[161:270]).all()
    assert torch.equal(got[:160], clean[:160]) and torch.equal(got[270:], clean[270:])
