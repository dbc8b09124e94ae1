"""GPU parity of multi-query scoring whose key units are cut into runs over
several workgroups (dsa_score_queries with few queries and a long key set),
and of fp8 keys on the multi-query kernel.

Every query's row must equal the single-query kernel's (dsa_full_scores, whose
parity with the oracle test_gpu_scores.py checks) bit for bit, since both run
the same tile code in the same order, and one row is held to the float64 oracle
with that file's bound: fp32 summation error, 1e-5 of sum_h |w_h| ReLU(q_h.k).
"""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from dsa_amd import progressive_kernel as P
from dsa_amd import sidecar
from oracle import scores as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,queries,length,fp8", [
    (1, 4, 704, False),      # 11 units: one run
    (1, 4, 768, False),      # 12 units: two halves
    (1, 9, 960, True),       # 15 units: eight and seven, with fp8 keys one query at a time
    (3, 64, 960, True),      # and four at a time
    (1, 1540, 960, False),   # 385 blocks: both halves would not be resident, one run
    (1, 4, 1023, False),     # 16 units: two runs of eight
    (1, 5, 1088, False),     # 17 units: a run of nine and one of eight; three idle waves in the second block
    (3, 130, 2049, False),   # causal limits inside several runs
    (1, 1540, 1100, False),  # 385 blocks: causal two runs by the units, three by the grid; without a limit one
    (1, 1540, 1472, False),  # 23 units: likewise, two runs by the units
    (1, 1540, 1473, False),  # 24 units: three runs with or without
    (1, 2100, 4096, False),  # 525 blocks: two runs by the grid, eight by the units
    (1, 3100, 1100, False),  # 775 blocks: one run by the grid
    (1, 300, 256, True),     # fp8 of four units: four queries at a time, one run
    (1, 4, 257, True),       # five units: one query at a time
    (1, 4, 1024, True),      # fp8 of few units: likewise
    (1, 48, 4096, True),     # 3072 units, 288 workgroups one query at a time: four, eight runs
    (2, 9, 4099, True),      # two key sets, ragged length, likewise
    (1, 256, 1024, True),    # 256 workgroups of 16 units, the last such; then four at a time: two runs of eight
    (1, 257, 1024, True),
    (1, 66, 6200, True),
    (2, 130, 2049, True),    # two key sets, a unit of one key, causal limits inside several runs
])
def test_runs_equal_single_queries(device, batch, queries, length, fp8) -> None:
    print(f"prefill runs B={batch} Q={queries} L={length} fp8={fp8}", flush=True)
    gen = torch.Generator().manual_seed(31 + length)
    q = (torch.randn(batch, queries, 64, 128, generator=gen) / math.sqrt(128)).to(torch.bfloat16)
    w = torch.randn(batch, queries, 64, generator=gen) / 8
    raw = torch.randn(batch, length, 128, generator=gen)
    blocks = (length + 127) // 128
    scales = None
    if fp8:
        scales = 0.003 + 0.004 * torch.rand(batch, blocks, generator=gen)
        keys = (raw / scales.repeat_interleave(128, dim=1)[:, :length, None]).clamp(-448, 448).to(torch.float8_e4m3fn)
        wide = S.dequantize_fp8_blocks(keys, scales)
    else:
        keys = raw.to(torch.bfloat16)
        wide = keys.float().numpy()
    qd, wd, kd = q.to(device), w.to(device), keys.to(device)
    sd = None if scales is None else scales.to(device)
    dense = sidecar.score_encoded(qd, wd, kd, key_scales=sd)
    offset = max(0, length - queries) // 2
    causal = sidecar.score_encoded(qd, wd, kd, key_scales=sd, causal=True, causal_offset=offset)
    picks = sorted({0, 1, queries // 2, queries - 2, queries - 1})
    for b in range(batch):
        for t in picks:
            one = P.full_scores_hip(qd[b, t], wd[b, t], kd[b], key_scales=None if sd is None else sd[b])
            assert torch.equal(dense[b, t], one), (b, t)
            visible = min(length, t + offset + 1)
            assert torch.equal(causal[b, t, :visible], one[:visible]), (b, t)
            assert torch.isneginf(causal[b, t, visible:]).all(), (b, t)
    t = picks[-1]
    ref = S.relu_index_score(q[0, t].float().numpy(), wide[0], w[0, t].numpy())
    bound = 1e-5 * S.abs_weight_scale(q[0, t].float().numpy(), wide[0], w[0, t].numpy()) + 1e-6
    assert np.all(np.abs(dense[0, t].cpu().double().numpy() - ref) <= bound)
