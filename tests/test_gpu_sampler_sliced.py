"""Few-row sampling in slices against whole rows, and whole rows against the oracle.

Up to 128 rows are cut into slices (wkv_sample_sliced); test_gpu_sampler.py's few-row launches
therefore check that path against the oracle. Here the one-workgroup-per-row kernel is checked
against the oracle on the same rows, and the two against each other over the sizes where the
cutting can go wrong: vocabularies around one and two slices, slices that end inside a chunk,
unaligned rows, rows whose slices hold nothing finite, lists that overflow.
"""

import numpy as np
import pytest
import torch

from test_gpu_sampler import ROWS, _check_rows
from wavelet_amd import _lib, sample, synth

pytestmark = pytest.mark.gpu


@pytest.fixture
def whole_rows(monkeypatch):
    """Calls inside take the one-workgroup-per-row kernel."""
    def use():
        monkeypatch.setattr(_lib.load(), "wkv_sample_workspace_size", lambda batch, vocab: 0)
    return use


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
def test_sliced_equals_whole_rows(cuda, whole_rows, vocab, dtype):
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
    sliced = sample(x, **kw)
    full = sample(x, **{k: v for k, v in kw.items() if k not in ("top_k", "top_p")})  # every row over the whole row
    whole_rows()
    for got, ref in ((sliced, sample(x, **kw)),
                     (full, sample(x, **{k: v for k, v in kw.items() if k not in ("top_k", "top_p")}))):
        assert torch.equal(got[0], ref[0]) and torch.equal(got[2], ref[2]) and torch.equal(got[3], ref[3])
        torch.testing.assert_close(got[1], ref[1], atol=1e-5, rtol=1e-5)
    assert sliced[3][-1].item() == 0 and sliced[0][-4].item() == vocab - 1


def test_sliced_row_counts_and_graph(cuda, whole_rows):
    """1 to 129 rows (the cut changes with the count, and stops past 128) against whole rows, then a
    captured call, replayed with new logits in between."""
    V = 50000
    gen = torch.Generator(device=cuda)
    gen.manual_seed(3)
    x = torch.randn((129, V), generator=gen, device=cuda) * 5
    seeds = torch.arange(129, dtype=torch.int64, device=cuda)
    counts = (1, 2, 7, 33, 64, 100, 128, 129)
    got = [sample(x[:n], seeds=seeds[:n], return_mask=True) for n in counts]
    gotk = [sample(x[:n], top_k=20, top_p=0.9, seeds=seeds[:n], return_mask=True) for n in counts]
    static = x[:5].clone()
    k = torch.full((5,), 20, dtype=torch.int32, device=cuda)
    p = torch.full((5,), 0.9, device=cuda)
    words = (V + 31) // 32
    out = (torch.empty(5, dtype=torch.int64, device=cuda), torch.empty(5, device=cuda),
           torch.empty((5, words), dtype=torch.int32, device=cuda), torch.empty(5, dtype=torch.int32, device=cuda))
    call = lambda: sample(static, top_k=k, top_p=p, seeds=seeds[:5], return_mask=True, out=out)  # noqa: E731
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    replays = []
    for i in range(4):
        static.copy_(x[5 * i:5 * i + 5])
        graph.replay()
        torch.cuda.synchronize()
        replays.append([t.clone() for t in out])
    whole_rows()
    for n, g, gk in zip(counts, got, gotk):
        for a, kw in ((g, {}), (gk, dict(top_k=20, top_p=0.9))):
            b = sample(x[:n], seeds=seeds[:n], return_mask=True, **kw)
            assert torch.equal(a[0], b[0]) and torch.equal(a[2], b[2]) and torch.equal(a[3], b[3]), n
            torch.testing.assert_close(a[1], b[1], atol=1e-5, rtol=1e-5)
    for i, r in enumerate(replays):
        b = sample(x[5 * i:5 * i + 5], top_k=k, top_p=p, seeds=seeds[:5], return_mask=True)
        assert torch.equal(r[0], b[0]) and torch.equal(r[2], b[2]) and torch.equal(r[3], b[3]), f"replay {i}"
