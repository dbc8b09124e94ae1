"""The one-workgroup row top-k (topk_rows_kernel through metrics.topk) against
the oracle's stable_topk, bit for bit: the candidate bound from a full and from
a sampled histogram, its pairwise, binned and recounted resolutions, and the
counting-sorted output, at the edges of the kernel's element counts and on rows
whose scores share an offset, hold outliers, ties or -inf."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from dsa_amd import metrics
from oracle import topk as T

pytestmark = pytest.mark.gpu


def _row(kind: str, length: int, rng) -> np.ndarray:
    x = rng.normal(size=length).astype(np.float32)
    if kind == "offset":  # one binade: bins finer than the key's top bits
        return (np.float32(100) + x * np.float32(0.01)).astype(np.float32)
    if kind == "outlier":  # the range of two values hides the rest in a few bins
        x[rng.integers(length)] = np.float32(1e30)
        x[rng.integers(length)] = np.float32(-1e30)
    elif kind == "tied":  # every cut crowded: the radix select and its ties
        x = rng.integers(-2, 3, size=length).astype(np.float32)
        x[x == 0] = rng.choice(np.array([0.0, -0.0], dtype=np.float32), size=int((x == 0).sum()))
    elif kind == "equal":
        x[:] = np.float32(-3.5)
    elif kind == "sparse":  # fewer finite scores than k, and +inf
        x[rng.random(length) < 0.97] = -np.inf
        x[rng.integers(length)] = np.inf
    elif kind == "periodic":  # the sampled quarter holds none of the top scores
        x[np.arange(length) % 4 != 0] += np.float32(10)
    return x


@pytest.mark.parametrize("kind", ["normal", "offset", "outlier", "tied", "equal", "sparse", "periodic"])
@pytest.mark.parametrize("length,k", [(4095, 128), (4097, 130), (8192, 1), (8193, 2048), (16384, 2049), (16385, 100),
                                      (30001, 4096), (32768, 600)])
def test_rows_match_oracle(device, kind, length, k) -> None:
    print(f"topk rows kind={kind} L={length} k={k}", flush=True)
    rng = np.random.default_rng(length + k)
    host = np.stack([_row(kind, length, rng) for _ in range(17)])
    wide = torch.full((17, length + 3), float("inf"), device=device)
    wide[:, :length] = torch.from_numpy(host)
    x = wide[:, :length]
    lengths = np.full(17, length, dtype=np.int32)
    lengths[3], lengths[5], lengths[7], lengths[9] = 0, k, k + 1, length - 1
    lens = torch.from_numpy(np.minimum(lengths, length)).to(device)
    in_order, values = metrics.topk(x, k, sorted=False, row_lengths=lens, return_values=True)
    ranked = metrics.topk(x, k, sorted=True, row_lengths=lens).cpu().numpy()
    in_order, values = in_order.cpu().numpy(), values.cpu().numpy()
    for r in (0, 3, 5, 7, 9, 16):
        n = int(min(lengths[r], length))
        assert ranked[r].tolist() == T.topk_sorted_padded(host[r], k, n).tolist(), r
        want = T.topk_index_order(host[r], k, n)
        assert in_order[r].tolist() == want.tolist(), r
        chosen = want >= 0
        np.testing.assert_array_equal(values[r][chosen].view(np.uint32), host[r][want[chosen]].view(np.uint32))
        assert np.isneginf(values[r][~chosen]).all()


@pytest.mark.parametrize("length,k,keys", [
    (1000, 1000, 999),    # every element with a key, k the row
    (4100, 4096, 4095),   # one key short of k
    (4100, 4096, 4096),   # exactly k keys
    (5000, 2048, 3),      # far fewer, full histogram
    (20000, 100, 60),     # and a sampled one
    (32768, 2048, 0),     # a row of poison alone
    (40000, 300, 7),      # chunks and their merge
])
def test_rows_of_all_ones_bits_are_padded(device, length, k, keys) -> None:
    # The NaN 0xffffffff is the one value without an order key: never chosen,
    # the output padded with -1 and -inf after the elements that have one.
    print(f"topk all-ones bits L={length} k={k} keys={keys}", flush=True)
    rng = np.random.default_rng(length + keys)
    host = np.full((3, length), 0xFFFFFFFF, dtype=np.uint32).view(np.float32)
    for r in range(3):
        host[r, rng.permutation(length)[:keys]] = rng.normal(size=keys).astype(np.float32)
    x = torch.from_numpy(host).to(device)
    # (past 32768 elements index order takes the distributed select, which ranks these NaNs last instead)
    for by_rank in (True, False) if length <= metrics.MAX_ROW else (True,):
        idx, val = metrics.topk(x, k, sorted=by_rank, return_values=True)
        idx, val = idx.cpu().numpy(), val.cpu().numpy()
        for r in range(3):
            at = np.flatnonzero(~np.isnan(host[r]))
            order = T.topk_sorted_padded(host[r][at], k, at.size) if by_rank else T.topk_index_order(host[r][at], k, at.size)
            want = np.where(order >= 0, at[order] if at.size else -1, -1)
            assert idx[r].tolist() == want.tolist(), (r, by_rank)
            np.testing.assert_array_equal(val[r][want >= 0], host[r][want[want >= 0]])
            assert np.isneginf(val[r][want < 0]).all()


def _crowded_row(kind: str, length: int, rng) -> np.ndarray:
    x = rng.normal(size=length).astype(np.float32)
    if kind == "some_inf":
        x[rng.random(length) < 0.4] = -np.inf
    elif kind == "mostly_inf":
        x[rng.random(length) < 0.95] = -np.inf
    elif kind == "all_inf":
        x[:] = -np.inf
    elif kind == "steps":  # some twenty distinct values
        x = np.round(x * 3).astype(np.float32)
    elif kind == "low_nan":  # NaNs that rank below -inf, by their bits
        x[rng.random(length) < 0.9] = -np.inf
        at = rng.random(length) < 0.5
        x[at] = (np.uint32(0xFFC00000) + rng.integers(0, 9, size=int(at.sum())).astype(np.uint32)).view(np.float32)
    elif kind == "run":  # the top scores next to each other
        x[length // 3 : length // 3 + length // 4] += np.float32(8)
    return x


def _by_rank(row: np.ndarray) -> np.ndarray:
    """Positions by (value desc, index asc); NaNs of the sign bit below -inf, the larger pattern last."""

    bits = row.view(np.uint32).astype(np.int64)
    value = np.where(np.isnan(row), -np.inf, np.where(row == 0, 0.0, row.astype(np.float64)))
    return np.lexsort((np.arange(row.size), np.where(np.isnan(row), bits, 0), -value))


@pytest.mark.parametrize("kind", ["normal", "some_inf", "mostly_inf", "all_inf", "steps", "low_nan", "run"])
@pytest.mark.parametrize("length,k", [(1000, 1000), (1001, 999), (4096, 2048), (4095, 4094), (5000, 129), (8190, 4096),
                                      (16384, 16), (24001, 2048), (32768, 256), (32767, 4096)])
def test_crowded_cuts_match_oracle(device, kind, length, k) -> None:
    # Cuts at -inf or below, among equal scores inside a bin, and k near the
    # row: the bound's steps down, the counts inside a bin, and both outputs.
    print(f"topk crowded kind={kind} L={length} k={k}", flush=True)
    rng = np.random.default_rng(2 * length + k)
    host = np.stack([_crowded_row(kind, length, rng) for _ in range(3)])
    x = torch.from_numpy(host).to(device)
    for by_rank in (True, False):
        idx, val = metrics.topk(x, k, sorted=by_rank, return_values=True)
        idx, val = idx.cpu().numpy(), val.cpu().numpy()
        for r in range(3):
            want = _by_rank(host[r])[:k]
            if not by_rank:
                want = np.sort(want)
            assert idx[r].tolist() == want.tolist(), (r, by_rank)
            np.testing.assert_array_equal(val[r].view(np.uint32), host[r][want].view(np.uint32))


@pytest.mark.parametrize("kind", ["normal", "outlier", "infinite", "denormal", "skewed"])
@pytest.mark.parametrize("length,k", [(4096, 2048), (5000, 4096), (8192, 3000), (20000, 2048)])
def test_ranked_rows_across_zero(device, kind, length, k) -> None:
    # Ranked outputs whose scores lie on both sides of zero, binned by score:
    # values that crowd one bin, spans past the largest float or of denormals,
    # and infinities, which keep the key's bins.
    print(f"topk across zero kind={kind} L={length} k={k}", flush=True)
    rng = np.random.default_rng(3 * length + k)
    host = rng.normal(loc=0.3, size=(3, length)).astype(np.float32)
    if kind == "outlier":
        host[:, 17] = np.float32(1e30)
    elif kind == "infinite":
        host[0, 5], host[1, 6], host[2, 7] = np.inf, np.float32(3e38), -np.inf
        host[1, 8] = np.float32(-3e38)
    elif kind == "denormal":
        host = (host * np.float32(1e-39)).astype(np.float32)
    elif kind == "skewed":
        host = np.where(host > 0, host, host * np.float32(1e-6)).astype(np.float32)
        host[:, ::7] = 0.0
        host[:, 3::7] = -0.0
    x = torch.from_numpy(host).to(device)
    idx, val = metrics.topk(x, k, sorted=True, return_values=True)
    idx, val = idx.cpu().numpy(), val.cpu().numpy()
    for r in range(3):
        want = T.stable_topk(host[r], k)
        assert idx[r].tolist() == want.tolist(), r
        np.testing.assert_array_equal(val[r].view(np.uint32), host[r][want].view(np.uint32))
