"""fp32 scores on both sides of the split kernel's limits (768 tiles of 16 keys
over a batch of at most 256), ragged lengths and several sequences, against the float64
oracle within fp32 summation error (1e-5 of sum_h |w_h| ReLU(q_h.k), the bound
of test_gpu_scores.py)."""

from __future__ import annotations

import ctypes
import math

import numpy as np
import pytest
import torch

from dsa_amd import _lib
from oracle import scores as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,length", [(1, 1), (1, 15), (2, 17), (1, 4097), (3, 4096), (1, 12288), (1, 12289), (2, 6200)])
def test_f32_scores_match_oracle(device, batch, length) -> None:
    print(f"fp32 scores B={batch} L={length}", flush=True)
    gen = torch.Generator().manual_seed(length)
    q = torch.randn(batch, 64, 128, generator=gen) / math.sqrt(128)
    w = torch.randn(batch, 64, generator=gen) / 8
    keys = torch.randn(batch, length, 128, generator=gen)
    qd, wd, kd = q.to(device), w.to(device), keys.to(device)
    out = torch.full((batch * length + 64,), 7.0, device=device)
    _lib.call("dsa_full_scores", qd.data_ptr(), wd.data_ptr(), kd.data_ptr(), None, out.data_ptr(), batch, length,
              _lib.DTYPE_F32, ctypes.c_void_p(_lib.stream_of(out)))
    assert (out[batch * length :] == 7.0).all()  # nothing past the rows
    got = out[: batch * length].reshape(batch, length).cpu().double().numpy()
    for b in range(batch):
        ref = S.relu_index_score(q[b].numpy(), keys[b].numpy(), w[b].numpy())
        scale = S.abs_weight_scale(q[b].numpy(), keys[b].numpy(), w[b].numpy())
        assert np.all(np.abs(got[b] - ref) <= 1e-5 * scale + 1e-6), b


@pytest.mark.parametrize("batch,length", [(1, 12288), (3, 4096), (12, 1024), (48, 256), (7, 1700), (256, 48), (257, 40)])
def test_f32_scores_do_not_depend_on_the_call(device, batch, length) -> None:
    # The same queries and keys in one call, sequence by sequence, and beside
    # enough further keys that the other kernel takes them: the same bits.
    print(f"fp32 scores across calls B={batch} L={length}", flush=True)
    gen = torch.Generator().manual_seed(length + batch)
    q = (torch.randn(batch, 64, 128, generator=gen) / math.sqrt(128)).to(device)
    w = (torch.randn(batch, 64, generator=gen) / 8).to(device)
    keys = torch.randn(batch, length, 128, generator=gen).to(device)
    more = torch.cat([keys, keys.new_zeros(batch, 12304, 128)], dim=1) if batch < 8 else None

    def scores(queries, weights, k):
        out = torch.empty(k.shape[0], k.shape[1], device=device)
        _lib.call("dsa_full_scores", queries.data_ptr(), weights.data_ptr(), k.data_ptr(), None, out.data_ptr(), k.shape[0],
                  k.shape[1], _lib.DTYPE_F32, ctypes.c_void_p(_lib.stream_of(out)))
        return out

    whole = scores(q, w, keys)
    for b in sorted({0, batch // 2, batch - 1}):
        assert torch.equal(scores(q[b : b + 1], w[b : b + 1], keys[b : b + 1])[0], whole[b]), b
    if more is not None:
        assert torch.equal(scores(q, w, more)[:, :length], whole)
