"""The list select of a decode step on score rows drawn to take each of its
ways: the cut found in the fine bins, ties past what one wave ranks, a cut an
octave above every list's lowest bin or below one of them, lists longer than
the registers, a last chunk of one key, and k at or past the row; and on signed
rows, whose cut lies near zero, below it, or among equal keys inside a bin that
is counted again."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from dsa_amd import decode
from oracle import topk as T

pytestmark = pytest.mark.gpu


def score_rows(kind, batch, length, k, rng):
    base = rng.uniform(1.0, 2.0, size=(batch, length))
    if kind == "octaves":  # a factor of two every 40 ranks: the cut lies octaves above the lists' ends
        base = np.exp2(8.0 - rng.permuted(np.tile(np.arange(length) / 40.0, (batch, 1)), axis=1).clip(max=100.0))
    elif kind == "coarse":  # eight distinct scores
        base = np.floor(base * 8) / 8
    elif kind == "crowded":  # the top-k in one run of keys, its lists' lowest bins far above the others'
        start = length // 3
        base[:, start : start + k] += 30.0
    elif kind == "negative":  # most keys score zero, fewer than k above it
        base[:, rng.permutation(length)[: length - max(1, k // 2)]] = -1.0
    return base


@pytest.mark.parametrize("kind", ["even", "octaves", "coarse", "crowded", "negative"])
@pytest.mark.parametrize(
    "batch,length,k",
    [(1, 256, 64), (1, 257, 300), (1, 4097, 256), (3, 5000, 5000), (5, 20011, 2048), (2, 32769, 100), (4, 131071, 2048)],
)
def test_list_select_matches_stable_topk(device, kind, batch, length, k) -> None:
    print(f"list select kind={kind} B={batch} L={length} k={k}", flush=True)
    rng = np.random.default_rng(length + k)
    want = torch.from_numpy(score_rows(kind, batch, length, k, rng)).float()
    # One head scores hi + lo, the wanted score to 16 bits; the rest score 0.
    q = torch.zeros(batch, 64, 128)
    q[:, 0, :2] = 1.0
    w = torch.zeros(batch, 64)
    w[:, 0] = 1.0
    keys = torch.zeros(batch, length, 128, dtype=torch.bfloat16)
    keys[:, :, 0] = want.to(torch.bfloat16)
    keys[:, :, 1] = (want - keys[:, :, 0].float()).to(torch.bfloat16)
    idx, scores, vals = decode.indexer_topk(
        q.to(torch.bfloat16).to(device), w.to(device), keys.to(device), k, return_scores=True, return_values=True
    )
    idx, scores, vals = idx.cpu().numpy(), scores.cpu().numpy(), vals.cpu().numpy()
    for b in range(batch):
        expect = T.topk_index_order(scores[b], k)
        np.testing.assert_array_equal(idx[b], expect)
        chosen = expect >= 0
        np.testing.assert_array_equal(vals[b][chosen], scores[b][expect[chosen]])
        assert np.isneginf(vals[b][~chosen]).all()


def signed_rows(kind, batch, length, rng):
    x = rng.normal(size=(batch, length))
    if kind == "shifted":  # the cut of k = L / 2 far below zero
        x -= 3.0
    elif kind == "tight":  # one binade, all in a few of the lists' bins
        x = 1.0 + x * 2.0**-9
    elif kind == "outlier":  # two keys stretch the bins over every other score
        x[:, 0], x[:, length // 2] = 1e30, 1e-30
    elif kind == "steps":  # about 40 distinct scores: crowded at every width
        x = np.round(x * 8) / 8
    elif kind == "zeros":  # nine keys in ten score zero, where the cut falls
        x[rng.random(x.shape) < 0.9] = 0.0
    elif kind == "huge":  # lists that end near -1e30 under a cut near 1e30: the last of the coarse bins
        x = np.where(rng.random(x.shape) < 0.55, 1.0, -1.0) * 1e30 * (1.0 + np.abs(x))
    return x


@pytest.mark.parametrize("kind", ["normal", "shifted", "tight", "outlier", "steps", "zeros", "huge"])
@pytest.mark.parametrize(
    "batch,length,k",
    [(1, 1024, 512), (1, 4096, 2048), (2, 2050, 2049), (16, 1024, 1000), (4, 4096, 4096), (3, 5003, 2501), (5, 20011, 2048),
     (4, 30000, 4500)],
)
def test_signed_scores_match_stable_topk(device, kind, batch, length, k) -> None:
    print(f"list select signed kind={kind} B={batch} L={length} k={k}", flush=True)
    want = torch.from_numpy(signed_rows(kind, batch, length, np.random.default_rng(length + k))).float()
    # score = ReLU(x) - ReLU(-x) = x, x to 16 bits over two dims.
    q = torch.zeros(batch, 64, 128)
    q[:, 0, :2], q[:, 1, :2] = 1.0, -1.0
    w = torch.zeros(batch, 64)
    w[:, 0], w[:, 1] = 1.0, -1.0
    keys = torch.zeros(batch, length, 128, dtype=torch.bfloat16)
    keys[:, :, 0] = want.to(torch.bfloat16)
    keys[:, :, 1] = (want - keys[:, :, 0].float()).to(torch.bfloat16)
    idx, scores, vals = decode.indexer_topk(
        q.to(torch.bfloat16).to(device), w.to(device), keys.to(device), k, return_scores=True, return_values=True
    )
    idx, scores, vals = idx.cpu().numpy(), scores.cpu().numpy(), vals.cpu().numpy()
    assert (scores < 0).any() or kind == "tight"
    for b in range(batch):
        expect = T.topk_index_order(scores[b], k)
        np.testing.assert_array_equal(idx[b], expect)
        np.testing.assert_array_equal(vals[b], scores[b][expect])
