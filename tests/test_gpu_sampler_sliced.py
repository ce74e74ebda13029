"""Few-row sampling in slices against the oracle and against whole rows, and whole rows against the oracle.

Up to 128 rows of more than 40,960 logits that are drawn from the whole vocabulary (no top_k, top_p or
min_p given) are cut into slices (wkv_sample_sliced). Those calls are checked against the oracle, and
against the one-workgroup-per-row kernel over the sizes where the cutting can go wrong: slices that end
inside a chunk, unaligned rows, rows whose slices hold nothing finite. Rows under thresholds are checked
at the lengths of their lists.
"""

import numpy as np
import pytest
import torch

from oracle import sampler as S
from test_gpu_sampler import ROWS, _check_rows
from wavelet_amd import _lib, sample, synth
from wavelet_amd.sampler import seen_bitmap

pytestmark = pytest.mark.gpu


@pytest.fixture
def whole_rows(monkeypatch):
    """Calls inside take the one-workgroup-per-row kernel."""
    def use():
        monkeypatch.setattr(_lib.load(), "wkv_sample_workspace_size", lambda batch, vocab: 0)
    return use


@pytest.fixture
def sliced_calls(monkeypatch):
    """The calls that were cut into slices, counted."""
    calls = []
    lib = _lib.load()
    inner = lib.wkv_sample_sliced
    monkeypatch.setattr(lib, "wkv_sample_sliced", lambda *a: (calls.append(a), inner(*a))[1])
    return calls


@pytest.mark.parametrize("vocab,pad", [(40961, 0), (50000, 3), (65536 + 8, 1), (151936, 0), (300007, 5)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_sliced_rows_match_oracle(cuda, sliced_calls, vocab, pad, dtype):
    """Sampled and greedy rows with and without a penalty, at any alignment; rows whose one finite logit is in
    the first or the last slice, half empty rows, ties of the maximum in different slices, rows of NaN."""
    B = 9
    gen = torch.Generator(device=cuda)
    gen.manual_seed(vocab)
    buf = torch.full((B, vocab + pad), float("nan"), dtype=dtype, device=cuda)
    x = buf[:, :vocab]
    x.copy_(torch.randn((B, vocab), generator=gen, device=cuda) * 4)
    x[3] = -float("inf")
    x[3, vocab - 1] = -3.0
    x[4] = float("nan")
    x[4, 0] = 2.0
    x[5, : vocab // 2] = -float("inf")
    x[6, [7, vocab // 2, vocab - 2]] = 50.0
    x[8] = float("nan")
    temps = np.array([1.0, 0.7, 1.0, 0.9, 1.0, 0.0, 0.0, 1.0, 1.0], np.float32)
    pens = np.array([1.0, 1.3, 1.2, 1.0, 1.0, 1.3, 1.0, 0.8, 1.0], np.float32)
    rng = np.random.default_rng(vocab)
    seen_lists = [rng.integers(0, vocab, 300) for _ in range(B)]
    seeds = np.arange(B, dtype=np.int64) * 1000 + 17
    tokens, logprobs, mask, counts = sample(
        x, temperature=torch.from_numpy(temps).to(cuda), repetition_penalty=torch.from_numpy(pens).to(cuda),
        seen=torch.from_numpy(seen_bitmap(seen_lists, vocab)).to(cuda), seeds=torch.from_numpy(seeds).to(cuda), step=5,
        return_mask=True)
    assert len(sliced_calls) == 1
    xf = x.float().cpu().numpy()
    bits = (mask.cpu().numpy().view(np.uint32)[:, :, None] >> np.arange(32, dtype=np.uint32)) & 1
    bits = bits.reshape(B, -1)[:, :vocab].astype(bool)
    for r in range(B):
        seen = np.zeros(vocab, bool)
        seen[seen_lists[r]] = True
        tok, lp, kept, _ = S.sample_row(xf[r], temperature=temps[r], repetition_penalty=pens[r], seen=seen,
                                        seed=int(seeds[r]), step=5)
        np.testing.assert_array_equal(bits[r], kept, err_msg=f"row {r}")
        assert counts[r].item() == kept.sum() and tokens[r].item() == tok, f"row {r}"
        if kept.any():
            assert abs(logprobs[r].item() - lp) < 1e-4, f"row {r}"
        else:
            assert logprobs[r].item() == lp == -np.inf, f"row {r}"


@pytest.mark.parametrize("vocab", [151936, 32001, 1000])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_whole_rows_match_oracle(cuda, whole_rows, vocab, dtype):
    whole_rows()
    B = len(ROWS)
    x = (synth.normal(synth.stream_key("smpw", vocab, str(dtype)), B * vocab) * 4.0).astype(np.float32).reshape(B, vocab)
    rng = np.random.default_rng(vocab)
    seen_lists = [rng.integers(0, vocab, 64) for _ in range(B)]
    _check_rows(cuda, x, ROWS, seen_lists, np.arange(B, dtype=np.int64) * 1000 + 17, 5, dtype)


@pytest.mark.parametrize("vocab", [8192, 8193, 32001])
def test_list_lengths_around_the_ranked_select(cuda, vocab):
    """Lists of 127 to 257 entries under top_k alone (ranked up to 128, then by radix) and under top_k and
    top_p together (up to 256), with ties at the threshold; min_p alone below and above one chunk per thread."""
    rows = [(1.0, k, p, 0.0, 1.0) for k in (100, 127, 128, 129, 255, 256, 257) for p in (1.0, 0.9)]
    rows += [(1.0, 0, 1.0, 0.3, 1.0), (0.7, 0, 1.0, 1e-4, 1.2), (1.0, 0, 0.99, 0.0, 1.0), (1.0, 0, 0.9999, 0.0, 1.0)]
    x = (synth.normal(synth.stream_key("smpr", vocab), len(rows) * vocab) * 4.0).astype(np.float32).reshape(len(rows), vocab)
    x[::3] = np.round(x[::3] * 16) / 16  # ties
    rng = np.random.default_rng(vocab)
    _check_rows(cuda, x, rows, [rng.integers(0, vocab, 64) for _ in rows], np.arange(len(rows), dtype=np.int64) * 7 + 1,
                3, torch.float32)


# (temperature, top_k, top_p, min_p, repetition_penalty): every path of a row, and k at and past the
# number of waves of the slices
MIX = ROWS + [(1.0, 300, 1.0, 0.0, 1.0), (1.0, 5000, 0.9, 0.0, 1.0), (0.0, 50, 1.0, 0.0, 1.0), (1.0, 0, 0.999, 0.0, 1.0),
              (1.0, 0, 1.0, 1e-6, 1.0), (0.0, 0, 1.0, 0.2, 1.0)]


@pytest.mark.parametrize("vocab", [8191, 8192, 8193, 16385, 24577, 65536 + 8, 151936, 300007])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_sliced_equals_whole_rows(cuda, whole_rows, sliced_calls, vocab, dtype):
    """Tokens, masks and counts equal; logprobs to float rounding of the kept mass (1e-5). Rows start
    three elements apart from any alignment and the row's tail is NaN past the vocabulary."""
    B, pad = len(MIX) + 4, 3
    gen = torch.Generator(device=cuda)
    gen.manual_seed(vocab)
    buf = torch.full((B, vocab + pad), float("nan"), dtype=dtype, device=cuda)
    x = buf[:, :vocab]
    x.copy_(torch.randn((B, vocab), generator=gen, device=cuda) * 4)
    x[-4] = -float("inf")  # one finite token, in the last slice
    x[-4, vocab - 1] = -3.0
    x[-3, : vocab // 2] = -float("inf")  # half of the row's slices empty
    x[-2] = 1.5  # flat: every list overflows
    x[-1] = float("nan")  # nothing finite
    rows = MIX + [(0.7, 50, 0.9, 0.0, 1.0), (0.7, 50, 0.9, 0.0, 1.0), (1.0, 40, 0.9, 0.0, 1.0), (1.0, 0, 1.0, 0.0, 1.0)]
    cols = [np.array([r[i] for r in rows]) for i in range(5)]
    kw = dict(temperature=torch.tensor(cols[0], dtype=torch.float32, device=cuda),
              top_k=torch.tensor(cols[1], dtype=torch.int32, device=cuda),
              top_p=torch.tensor(cols[2], dtype=torch.float32, device=cuda),
              min_p=torch.tensor(cols[3], dtype=torch.float32, device=cuda),
              repetition_penalty=torch.tensor(cols[4], dtype=torch.float32, device=cuda),
              seen=torch.randint(-2 ** 31, 2 ** 31, (B, (vocab + 31) // 32), generator=gen, device=cuda).to(torch.int32),
              seeds=torch.arange(B, dtype=torch.int64, device=cuda) * 77 + 5, step=9, return_mask=True)
    listed = sample(x, **kw)  # every path of a whole row
    assert not sliced_calls
    uncut = {k: v for k, v in kw.items() if k not in ("top_k", "top_p", "min_p")}
    full = sample(x, **uncut)
    assert len(sliced_calls) == (vocab > 40960)
    whole_rows()
    for got, ref in ((listed, sample(x, **kw)), (full, sample(x, **uncut))):
        assert torch.equal(got[0], ref[0]) and torch.equal(got[2], ref[2]) and torch.equal(got[3], ref[3])
        torch.testing.assert_close(got[1], ref[1], atol=1e-5, rtol=1e-5)
    assert len(sliced_calls) == (vocab > 40960)
    for got in (listed, full):
        assert got[3][-1].item() == 0 and got[0][-4].item() == vocab - 1


def test_sliced_row_counts_and_graph(cuda, whole_rows, sliced_calls):
    """1 to 129 rows (the cut changes with the count, and stops where a slice is too little shorter than the
    row, here between 65 and 100 rows, and past 128 anywhere) against whole rows, then captured calls, in slices and under
    thresholds, replayed with new logits in between."""
    V = 50000
    gen = torch.Generator(device=cuda)
    gen.manual_seed(3)
    x = torch.randn((129, V), generator=gen, device=cuda) * 5
    seeds = torch.arange(129, dtype=torch.int64, device=cuda)
    counts = (1, 2, 7, 33, 64, 100, 128, 129)
    got = [sample(x[:n], seeds=seeds[:n], return_mask=True) for n in counts]
    lib = _lib.load()
    assert len(sliced_calls) == sum(lib.wkv_sample_workspace_size(n, V) > 0 for n in counts) >= 5
    assert lib.wkv_sample_workspace_size(129, 151936) == 0 < lib.wkv_sample_workspace_size(128, 151936)
    gotk = [sample(x[:n], top_k=20, top_p=0.9, seeds=seeds[:n], return_mask=True) for n in counts]
    static = x[:5].clone()
    k = torch.full((5,), 20, dtype=torch.int32, device=cuda)
    p = torch.full((5,), 0.9, device=cuda)
    words = (V + 31) // 32
    replays = {}
    for name, args in (("sliced", {}), ("lists", dict(top_k=k, top_p=p))):
        out = (torch.empty(5, dtype=torch.int64, device=cuda), torch.empty(5, device=cuda),
               torch.empty((5, words), dtype=torch.int32, device=cuda), torch.empty(5, dtype=torch.int32, device=cuda))
        call = lambda: sample(static, seeds=seeds[:5], return_mask=True, out=out, **args)  # noqa: B023,E731
        before = len(sliced_calls)
        call()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            call()
        assert len(sliced_calls) - before == (2 if name == "sliced" else 0)
        replays[name] = []
        for i in range(4):
            static.copy_(x[5 * i:5 * i + 5])
            graph.replay()
            torch.cuda.synchronize()
            replays[name].append([t.clone() for t in out])
            sample(x[:3], seeds=seeds[:3])  # the program's own eager work in between
    whole_rows()
    for n, g, gk in zip(counts, got, gotk):
        for a, kw in ((g, {}), (gk, dict(top_k=20, top_p=0.9))):
            b = sample(x[:n], seeds=seeds[:n], return_mask=True, **kw)
            assert torch.equal(a[0], b[0]) and torch.equal(a[2], b[2]) and torch.equal(a[3], b[3]), n
            torch.testing.assert_close(a[1], b[1], atol=1e-5, rtol=1e-5)
    for name, args in (("sliced", {}), ("lists", dict(top_k=k, top_p=p))):
        for i, r in enumerate(replays[name]):
            b = sample(x[5 * i:5 * i + 5], seeds=seeds[:5], return_mask=True, **args)
            assert torch.equal(r[0], b[0]) and torch.equal(r[2], b[2]) and torch.equal(r[3], b[3]), f"{name} replay {i}"
            torch.testing.assert_close(r[1], b[1], atol=1e-5, rtol=1e-5)
