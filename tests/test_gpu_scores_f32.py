"""fp32 scores on both sides of the split kernel's tile limit (768 tiles of 16
keys over the batch), ragged lengths and several sequences, against the float64
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
