"""Prefill launch grids: how query heads and tiles are packed into workgroups, by the sizes.
Against the float64 oracle."""

import pytest

from test_gpu_prefill import _case, _run_and_check

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
