"""The dynamic step's replay at the edges of what its threads keep in
registers: k around the 2048 keys read first, and one key of k, with blocks
that make the waves' listed keys share a group or not.  Every result equals
the sequential scan's."""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from dsa_amd import decode, temporal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 2047, 2048, 2049, 3001])
@pytest.mark.parametrize("block,wave", [(16, 1), (64, 9)])
def test_replay_key_counts(device, monkeypatch, k, block, wave) -> None:
    print(f"replay keys k={k} bs={block} W={wave}", flush=True)
    gen = torch.Generator().manual_seed(k + block)
    batch, length = 2, 6003
    q = (torch.randn(batch, 64, 128, generator=gen) / math.sqrt(128)).to(torch.bfloat16)
    q_next = (q.float() + 0.05 * torch.randn(batch, 64, 128, generator=gen) / math.sqrt(128)).to(torch.bfloat16)
    w = torch.randn(batch, 64, generator=gen) / 8
    keys = torch.randn(batch, length, 128, generator=gen).to(torch.bfloat16).to(device)
    q, q_next, w = q.to(device), q_next.to(device), w.to(device)
    prev_topk, prev_scores = decode.indexer_topk(q, w, keys[:, : length - 1].contiguous(), k, return_scores=True)
    prev_max = temporal.block_max(prev_scores, block)
    gamma = torch.full((batch,), -0.25 * float(prev_scores.std()), device=device)

    def run():
        s = temporal.temporal_step(q_next, w, keys, prev_max, length - 1, prev_topk, gamma, block_size=block,
                                   method="dynamic", scan_order="previous_hot", wave=wave)
        return [x.cpu().numpy() for x in (s.scores, s.evaluated_blocks, s.qk_scored, s.topk)]

    monkeypatch.setenv("DSA_AMD_TEMPORAL_PATH", "launch")
    want = run()
    monkeypatch.delenv("DSA_AMD_TEMPORAL_PATH")
    for splits in (None, "0.25", "0.05,0.4"):
        if splits:
            monkeypatch.setenv("DSA_AMD_TEMPORAL_ROUNDS", splits)
        for got, expect in zip(run(), want):
            np.testing.assert_array_equal(got, expect)
