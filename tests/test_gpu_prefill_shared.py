"""GPU parity of the shared-grid prefill (wkv_prefill_gqa_shared) against the float64 oracle.

The number of workgroups that share the launch's 64-key steps is forced here: from eight (whole
query tiles in the middle of a workgroup's share, one wrapping to the next KV head) to more than
there are steps (every part one step, workgroups without work), so that parts end on the causal
diagonal, inside a block, past a query's last key and at the context's end. Tolerances as for
the plain prefill; the workspace is exactly the size the library asks for, between poisoned pads.
"""

import ctypes

import numpy as np
import pytest
import torch

from kvcase import Guarded, assert_guards, bits_of, check_attention, to_dev_bits
from oracle import fp8, paged
from test_gpu_prefill import _case
from wavelet_amd import _lib
from wavelet_amd.cache import KV_DTYPES

pytestmark = pytest.mark.gpu

BF16 = torch.bfloat16


def _shared_call(cuda, w, cache, new, workgroups, sinks=None):
    """wkv_prefill_gqa_shared over the case, appending; the workspace guarded."""
    kn, vn, q, nslots, cu = new
    lib = _lib.load()
    qd, kd, vd = (to_dev_bits(x, BF16, cuda) for x in (q, kn, vn))
    bt, sl = torch.from_numpy(w.block_tables).to(cuda), torch.from_numpy(w.context_lens).to(cuda)
    cud, slots = torch.from_numpy(cu).to(cuda), torch.from_numpy(nslots).to(cuda)
    sd = None if sinks is None else torch.from_numpy(sinks).to(cuda)
    out = torch.full(qd.shape, float("nan"), dtype=BF16, device=cuda)
    mql, msl = int(np.diff(cu).max()), int(w.context_lens.max())
    need = lib.wkv_prefill_workspace_size(w.batch, KV_DTYPES[cache.kv_dtype], w.num_kv_heads, w.num_q_heads, w.head_dim, mql, msl, workgroups)
    ws = Guarded((max(need, 16),), torch.uint8, cuda)
    args = [ctypes.byref(cache.descriptor()), kd.data_ptr(), kd.stride(0), kd.stride(1), vd.data_ptr(), vd.stride(0),
            vd.stride(1), slots.data_ptr(), len(nslots), qd.data_ptr(), qd.stride(0), qd.stride(1), out.data_ptr(),
            out.stride(0), out.stride(1), w.num_q_heads, cud.data_ptr(), sl.data_ptr(), bt.data_ptr(), bt.stride(0),
            bt.shape[1], w.batch, mql, msl, float(w.scale), workgroups]
    stream = torch.cuda.current_stream(cuda).cuda_stream
    sp = None if sd is None else sd.data_ptr()
    if need > 0:  # a workspace one byte short is refused before any launch, the append's among them
        before = cache.k.clone(), cache.v.clone()
        assert lib.wkv_prefill_gqa_shared(*args, ws.t.data_ptr(), need - 1, sp, stream) == _lib.WKV_ERR_INVALID
        for x, y in zip(before, (cache.k, cache.v)):
            assert torch.equal(x.view(torch.uint8), y.view(torch.uint8))
    _lib.check(lib.wkv_prefill_gqa_shared(*args, ws.t.data_ptr(), need, sp, stream), "shared prefill")
    assert_guards([ws], "shared prefill")
    return out, need


def _reference(w, cache, host, new, sinks=None):
    kc, vc, ks, vs = host
    kn, vn, q, nslots, cu = new
    if ks is not None:
        paged.append_fp8(kc, vc, ks, vs, kn, vn, nslots)
        kf = fp8.dequantize(paged.k_logical(kc).reshape(w.num_blocks, w.block_size, w.num_kv_heads, w.head_dim),
                            ks[:, None, :, None])
        vf = fp8.dequantize(paged.v_logical(vc), vs[:, None, :, None])
    else:
        paged.append_bf16(kc, vc, kn, vn, nslots)
        kl, vl = paged.logical_kv(kc, vc)
        kf, vf = paged.bf16_to_f32(kl), paged.bf16_to_f32(vl)
    return paged.prefill_gqa(paged.bf16_to_f32(q), kf, vf, w.block_tables, w.context_lens, cu, w.scale, sinks=sinks)


# (new tokens, total length): whole prompts, chunks after context, one token, none; a context of
# 64 k keys exactly and one key more
MIX = ([37, 16, 1, 130, 0, 64, 1, 33], [37, 300, 50, 700, 20, 64, 641, 320])


@pytest.mark.parametrize("workgroups", [8, 37, 512])
@pytest.mark.parametrize("kv_dtype", ["bf16", "fp8_e4m3"])
@pytest.mark.parametrize("hq,hkv,d,bs", [(32, 8, 128, 16), (14, 2, 64, 16), (28, 4, 128, 32), (16, 8, 128, 16),
                                         (3, 3, 64, 256), (5, 1, 128, 48)])
def test_prefill_shared_matches_oracle(cuda, hq, hkv, d, bs, kv_dtype, workgroups):
    name = f"pfshare{hq}{hkv}{d}{bs}"
    w, cache, host, new = _case(cuda, name, hq, hkv, d, bs, *MIX, kv_dtype)
    out, need = _shared_call(cuda, w, cache, new, workgroups)
    assert need > 0
    check_attention(paged.bf16_to_f32(bits_of(out)), _reference(w, cache, host, new), f"{name} {workgroups}")


def test_prefill_shared_with_sinks_and_a_long_context(cuda):
    """Sinks join the merged denominator once; a 9,000-token context crosses the 64-block table window
    inside a part and between parts."""
    w, cache, host, new = _case(cuda, "pfsharelong", 14, 2, 64, 16, [50, 7, 1], [9000, 2100, 4097], "bf16")
    sinks = np.linspace(-3, 9, 14).astype(np.float32)
    sinks[0] = -np.inf
    out, _ = _shared_call(cuda, w, cache, new, 24, sinks=sinks)
    check_attention(paged.bf16_to_f32(bits_of(out)), _reference(w, cache, host, new, sinks), "sinks")


def test_prefill_shared_of_very_negative_scores(cuda):
    """A part that a query does not see must not set its merged maximum: every score is far below
    zero, and the parts past the diagonal hold no key of the early queries."""
    w, cache, host, new = _case(cuda, "pfshareneg", 8, 2, 64, 16, [200, 90], [200, 90], "bf16")
    kn, vn, q, nslots, cu = new
    kn = paged.bf16_to_f32(kn) * 0 + 8.0  # scores -8 * 8 * 64 / 8 = -512
    q = paged.bf16_to_f32(q) * 0.01 - 8.0
    new = (synth_bits(kn), vn, synth_bits(q), nslots, cu)
    out, need = _shared_call(cuda, w, cache, new, 96)
    assert need > 0
    check_attention(paged.bf16_to_f32(bits_of(out)), _reference(w, cache, host, new), "negative scores")


def synth_bits(x):
    from wavelet_amd import synth

    return synth.to_bf16_bits(x)
