"""Prefill launch grids: how query heads and tiles are packed into workgroups, and when a launch
shares its keys, by the sizes and length bounds the caller gives. Against the float64 oracle."""

import numpy as np
import pytest
import torch

from kvcase import bits_of, check_attention, to_dev_bits
from oracle import fp8, paged
from test_gpu_prefill import BF16, _case, _run_and_check
from test_gpu_prefill_shared import _reference, _shared_call
from wavelet_amd import PagedKVCache, _lib, prefill_gqa
from wavelet_amd.cache import KV_DTYPES
from wavelet_amd.plan import PrefillStep

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv_dtype", ["bf16", "fp8_e4m3"])
@pytest.mark.parametrize("hq,hkv,d,qlens,ctx", [
    (14, 2, 64, [255, 64, 1, 33, 256, 200, 31, 100], 0),  # 256 groups of a tile's heads: a tile to itself
    (14, 2, 64, [257, 64, 1, 33, 256, 200, 31, 100], 0),  # 288
    (14, 2, 64, [512, 64, 1, 33, 256, 200, 31, 100], 0),  # 512
    (14, 2, 64, [513, 64, 1, 33, 256, 200, 31, 100], 0),  # 544: packed across tiles
    (16, 8, 128, [256, 1, 90, 17], 48),
    (16, 8, 128, [257, 1, 90, 17], 48),
    (5, 1, 128, [289, 0, 128, 7] * 4, 20),
    (8, 2, 64, [300, 1, 100, 60, 290, 33, 7, 256] * 4, 0),  # 768 workgroups: an XCD's sub-items in turn
    (8, 2, 64, [400, 1, 100, 60, 290, 33, 7, 256] * 4, 0),  # 1,024: one after another
])
def test_both_sides_of_the_packing_bounds(cuda, hq, hkv, d, qlens, ctx, kv_dtype):
    w, cache, host, new = _case(cuda, f"pfgrid{hq}{d}{max(qlens)}", hq, hkv, d, 16, qlens, [n + ctx + 1 for n in qlens],
                                kv_dtype)
    _run_and_check(cuda, w, cache, host, new, f"{hq}/{hkv} {max(qlens)}")


@pytest.mark.parametrize("kv_dtype", ["bf16", "fp8_e4m3"])
@pytest.mark.parametrize("hq,hkv,d,n_seq,shared", [(14, 2, 64, 8, 0), (14, 2, 64, 16, 0), (16, 8, 128, 4, 0),
                                                   (5, 1, 128, 16, 0), (3, 3, 64, 1, 0), (14, 2, 64, 2, 24), (3, 1, 128, 2, 96),
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


def _need(w, cache, cu, keys):
    return _lib.load().wkv_prefill_workspace_size(w.batch, KV_DTYPES[cache.kv_dtype], w.num_kv_heads, w.num_q_heads,
                                                  w.head_dim, int(np.diff(cu).max()), keys, 0)


@pytest.mark.parametrize("sinks", [False, True])
@pytest.mark.parametrize("kv_dtype", ["bf16", "fp8_e4m3"])
@pytest.mark.parametrize("hq,hkv,d,qlens,lens", [(28, 4, 128, [1, 1, 1], [5000, 4096, 3000]),
                                                 (14, 2, 64, [70, 33, 1], [4000, 700, 2049]),
                                                 (32, 8, 128, [40, 0], [3000, 64])])
def test_launches_shared_by_the_librarys_choice(cuda, hq, hkv, d, qlens, lens, kv_dtype, sinks):
    w, cache, host, new = _case(cuda, f"pfauto{hq}{d}", hq, hkv, d, 16, qlens, lens, kv_dtype)
    assert _need(w, cache, new[4], max(lens)) > 0
    if not sinks:
        _run_and_check(cuda, w, cache, host, new, f"auto {hq}/{hkv}")
        return
    s = np.linspace(-2, 12, hq).astype(np.float32)
    kn, vn, q, nslots, cu = new
    out = prefill_gqa(to_dev_bits(q, BF16, cuda), cache, torch.from_numpy(w.block_tables).to(cuda),
                      torch.from_numpy(w.context_lens).to(cuda), torch.from_numpy(cu).to(cuda), w.scale,
                      key=to_dev_bits(kn, BF16, cuda), value=to_dev_bits(vn, BF16, cuda),
                      slot_mapping=torch.from_numpy(nslots).to(cuda), sinks=torch.from_numpy(s).to(cuda))
    ref = _reference(w, cache, host, new, s)
    plain = paged.prefill_gqa(paged.bf16_to_f32(q), *_logical(host), w.block_tables, w.context_lens, cu, w.scale)
    # (over thousands of keys the outputs are small: what the sinks change is a part of them, ten
    # times the relative tolerance or more)
    assert np.linalg.norm(ref - plain) > 0.1 * np.linalg.norm(plain)
    check_attention(paged.bf16_to_f32(bits_of(out)), ref, f"auto sinks {hq}/{hkv}")


def _logical(host):
    kc, vc, ks, vs = host
    if ks is None:
        return tuple(paged.bf16_to_f32(x) for x in paged.logical_kv(kc, vc))
    shape = (len(ks), kc.shape[3], kc.shape[1], kc.shape[2] * kc.shape[4])
    return (fp8.dequantize(paged.k_logical(kc).reshape(shape), ks[:, None, :, None]),
            fp8.dequantize(paged.v_logical(vc), vs[:, None, :, None]))


@pytest.mark.parametrize("kv_dtype", ["bf16", "fp8_e4m3"])
def test_layers_of_a_plan_take_turns_with_its_workspace(cuda, kv_dtype):
    """Three layers of different contents (and of two head layouts) over one plan, shared by the library's
    choice, run twice."""
    qlens, lens = [3, 50, 1], [4000, 2500, 3000]
    layers = [_case(cuda, "pfplan", hq, hkv, 128, 16, qlens, lens, kv_dtype) for hq, hkv in [(28, 4), (16, 4), (28, 4)]]
    wl, cache, host, (kn, vn, q, nslots, cu) = layers[2]
    layers[2] = wl, cache, host, (vn, kn, q ^ np.uint16(0x8000), nslots, cu)
    w, _, _, (_, _, _, nslots, cu) = layers[0]
    dev = [[to_dev_bits(new[i], BF16, cuda) for _, _, _, new in layers] for i in (2, 0, 1)]  # q, key, value
    outs = [torch.full_like(q, float("nan")) for q in dev[0]]
    assert all(_need(x[0], x[1], cu, max(lens)) > 0 for x in layers)
    assert all(np.array_equal(x[0].block_tables, w.block_tables) for x in layers)
    step = PrefillStep([x[1] for x in layers], dev[0], dev[1], dev[2], outs, torch.from_numpy(w.block_tables).to(cuda),
                       torch.from_numpy(w.context_lens).to(cuda), torch.from_numpy(cu).to(cuda),
                       torch.from_numpy(nslots).to(cuda), w.scale, max(qlens), max(lens))
    for _ in range(2):
        step.run()
    for i, (wl, cache, host, new) in enumerate(layers):
        check_attention(paged.bf16_to_f32(bits_of(outs[i])), _reference(wl, cache, host, new), f"layer {i}")


def test_layers_of_different_block_sizes_share_a_plan(cuda):
    """One table over caches of 16- and 64-token blocks: the second layer's launch sees four times the keys, and
    the plan's workspace is sized for it."""
    gen = torch.Generator(device=cuda)
    gen.manual_seed(1)
    rnd = lambda *shape: torch.randn(shape, generator=gen, device=cuda).to(BF16)  # noqa: E731
    caches = [PagedKVCache(100, bs, 8, 128, device=cuda) for bs in (16, 64)]
    for c in caches:
        c.k.copy_(rnd(*c.k.shape))
        c.v.copy_(rnd(*c.v.shape))
    q, k, v = ([rnd(1, h, 128) for _ in caches] for h in (32, 8, 8))
    outs = [torch.empty_like(x) for x in q]
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device=cuda)  # noqa: E731
    bt = torch.arange(100, dtype=torch.int32, device=cuda).view(1, 100)
    slots = torch.tensor([1499], device=cuda)
    needs = [_lib.load().wkv_prefill_workspace_size(1, 0, 8, 32, 128, 1, min(6000, 100 * c.block_size), 0) for c in caches]
    assert 0 < needs[0] < needs[1]
    step = PrefillStep(caches, q, k, v, outs, bt, i32(1500), i32(0, 1), slots, 0.1, 1, 6000)
    step.run()
    for c, qq, oo in zip(caches, q, outs):
        assert torch.equal(oo, prefill_gqa(qq, c, bt, i32(1500), i32(0, 1), 0.1, max_query_len=1, max_seq_len=6000))


@pytest.mark.parametrize("kv_dtype", ["bf16", "fp8_e4m3"])
@pytest.mark.parametrize("hq,hkv,d,qlens,lens", [(32, 8, 128, [200], [200]), (14, 2, 64, [60, 1, 0, 33], [260, 3, 40, 33]),
                                                 (28, 4, 128, [37, 250, 1], [37, 250, 900]),
                                                 (28, 4, 128, [16, 1], [6000, 300]), (16, 8, 128, [0, 1], [5, 70])])
def test_length_bounds_above_the_lengths(cuda, hq, hkv, d, qlens, lens, kv_dtype):
    """A caller that gives the model's limit for max_seq_len gets a launch that could share; what it does
    follows the lengths on the device. Where that is whole unit groups, the bits are the plain launch's."""
    w, cache, host, new = _case(cuda, f"pfbound{hq}{len(qlens)}", hq, hkv, d, 16, qlens, lens, kv_dtype)
    kn, vn, q, nslots, cu = new
    bt = torch.full((w.batch, 16384 // 16), -1, dtype=torch.int32, device=cuda)
    bt[:, :w.block_tables.shape[1]] = torch.from_numpy(w.block_tables).to(cuda)
    args = (to_dev_bits(q, BF16, cuda), cache, bt, torch.from_numpy(w.context_lens).to(cuda),
            torch.from_numpy(cu).to(cuda), w.scale)
    assert _need(w, cache, cu, 16384) > 0
    cache.append(to_dev_bits(kn, BF16, cuda), to_dev_bits(vn, BF16, cuda), torch.from_numpy(nslots).to(cuda))
    mql = max(qlens)
    out = torch.full((len(q), hq, d), float("nan"), dtype=BF16, device=cuda)
    prefill_gqa(*args, max_query_len=mql, max_seq_len=16384, out=out)
    check_attention(paged.bf16_to_f32(bits_of(out)), _reference(w, cache, host, new), "bounds")
    if max(lens) <= 300:
        assert torch.equal(out, prefill_gqa(*args, max_query_len=mql, max_seq_len=max(lens)))
