"""Rows whose largest logit is +inf, on every path of the sampler, against the oracle.

Such a row has no distances below its maximum (inf - inf is NaN), so the ranges and bins that the
capture passes work with cannot hold its maximum: the whole row decides by key alone.
"""

import numpy as np
import pytest
import torch

from oracle import sampler as S
from wavelet_amd import sample, synth
from wavelet_amd.sampler import seen_bitmap

pytestmark = pytest.mark.gpu

# (temperature, top_k, top_p, min_p, repetition_penalty)
ROWS = [(1.0, 0, 1.0, 0.1, 1.0), (0.0, 0, 1.0, 0.1, 1.3), (0.7, 0, 1.0, 1e-6, 1.2), (1.0, 0, 0.9, 0.0, 1.0),
        (0.8, 0, 0.3, 0.0, 1.3), (0.0, 0, 0.9, 0.05, 1.0), (1.0, 1, 1.0, 0.0, 1.0), (1.0, 50, 1.0, 0.0, 1.0),
        (0.7, 2000, 0.9, 0.0, 1.1), (1.0, 50, 0.9, 0.05, 1.0), (1.0, 0, 1.0, 0.0, 1.0), (0.0, 0, 1.0, 0.0, 1.0)]


@pytest.mark.parametrize("vocab", [1000, 50000, 151936, 270000])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_with_an_infinite_maximum(cuda, vocab, dtype):
    """One, two and 5,000 infinite logits (at both ends of the row; more than the list holds), finite ones
    at the type's largest magnitude beside them; some rows hold nothing else but -inf."""
    B = len(ROWS)
    x = (synth.normal(synth.stream_key("smpinf", vocab), B * vocab) * 4.0).astype(np.float32).reshape(B, vocab)
    x = torch.from_numpy(x).to(dtype)
    big = torch.finfo(dtype).max
    x[:, 5], x[:, 6], x[:, 7] = big, -big, float("nan")
    at = [[0], [vocab - 1], [3, vocab - 2], [0, vocab - 1], list(range(0, min(vocab, 10000), 2))]
    for r in range(B):
        if r % 4 == 3:
            x[r] = -float("inf")
        x[r, at[r % len(at)]] = float("inf")
    rng = np.random.default_rng(vocab)
    seen_lists = [np.concatenate([rng.integers(0, vocab, 64), at[r % len(at)][:1]]) for r in range(B)]
    cols = [np.array([r[i] for r in ROWS]) for i in range(5)]
    seeds = np.arange(B, dtype=np.int64) * 31 + 7
    kw = dict(temperature=torch.tensor(cols[0], dtype=torch.float32, device=cuda),
              repetition_penalty=torch.tensor(cols[4], dtype=torch.float32, device=cuda),
              seen=torch.from_numpy(seen_bitmap(seen_lists, vocab)).to(cuda), seeds=torch.from_numpy(seeds).to(cuda),
              step=3, return_mask=True)
    per_row = {"top_k": torch.tensor(cols[1], dtype=torch.int32, device=cuda),
               "top_p": torch.tensor(cols[2], dtype=torch.float32, device=cuda),
               "min_p": torch.tensor(cols[3], dtype=torch.float32, device=cuda)}
    logits = x.to(cuda)
    xf = x.to(torch.float32).numpy()
    for given in (("top_k", "top_p", "min_p"), ("min_p",), ("top_p",), ("top_k",), ()):
        tokens, logprobs, mask, counts = sample(logits, **kw, **{n: per_row[n] for n in given})
        bits = (mask.cpu().numpy().view(np.uint32)[:, :, None] >> np.arange(32, dtype=np.uint32)) & 1
        bits = bits.reshape(B, -1)[:, :vocab].astype(bool)
        for r in range(B):
            seen = np.zeros(vocab, bool)
            seen[seen_lists[r]] = True
            opt = {n: cols[i][r] for i, n in ((1, "top_k"), (2, "top_p"), (3, "min_p")) if n in given}
            with np.errstate(over="ignore"):  # (the largest logits scale past the type)
                tok, lp, kept, amb = S.sample_row(xf[r], temperature=cols[0][r], repetition_penalty=cols[4][r],
                                                  seen=seen, seed=int(seeds[r]), step=3, **opt)
            name = f"row {r} {ROWS[r]} given {given}"
            assert not amb and np.isnan(lp), name
            assert tokens[r].item() == tok, name
            np.testing.assert_array_equal(bits[r], kept, err_msg=name)
            assert counts[r].item() == kept.sum(), name
            assert torch.isnan(logprobs[r]).item(), name
