"""Sidecar indexer: encoders and batched / multi-query scoring.

Reference: ``temporal_dsa/sidecar.py``.
  * ``apply_noninterleaved_rope`` (sidecar.py:10-28) and the encoders of
    ``LightningIndexerSidecar`` (sidecar.py:31-88): the projections wq / wk /
    weights_proj run in the library's own kernels, a weight-streaming kernel
    for a decode step (``dsa_project_rows``) and an MFMA GEMM for larger
    batches (``dsa_project_gemm``); the LayerNorm, RoPE, head-weight scaling
    and the key-cache append after them run in one HIP pass per row
    (``dsa_encode_keys_epilogue``, ``dsa_encode_queries_epilogue``,
    ``dsa_rope``), with torch's per-op rounding in the row dtype, or, for
    the queries of a bf16 batch, inside the GEMM's output stage.  The module
    runs in its parameter dtype (fp32 or bf16); autocast's mixed flow is not
    reproduced.
  * ``score_encoded`` (sidecar.py:89-107): ``[B,Q,H,D] x [B,K,D] -> [B,Q,K]``
    fp32, ``ReLU(q.k) * w`` summed over heads.

Differences of ``score_encoded`` from the reference, all documented at the call:
  * dots stay fp32 (the reference's bf16 einsum rounds each dot to bf16 before
    the ReLU; both agree within the 1e-2 relative bf16 tolerance);
  * ``causal=True`` masks key j of query t unless ``j <= t + causal_offset``
    (masked scores are -inf); the reference has no mask;
  * fp8 e4m3fn keys with one fp32 scale per 128 keys are accepted through
    ``key_scales`` ``[B, ceil(K/128)]``.
The KL loss and the teacher target (sidecar.py:123-137) belong to training
and are not part of this package.
"""

from __future__ import annotations

import math

import torch
from torch import nn

from . import _lib
from .progressive_kernel import HEAD_DIM, HEADS

_ROW_DTYPES = {torch.float32: _lib.DTYPE_F32, torch.bfloat16: _lib.DTYPE_BF16}


def score_encoded(
    queries: torch.Tensor,
    weights: torch.Tensor,
    keys: torch.Tensor,
    *,
    key_chunk_size: int | None = None,
    causal: bool = False,
    causal_offset: int | None = None,
    key_scales: torch.Tensor | None = None,
) -> torch.Tensor:
    """Indexer scores of every (query, key) pair, fp32 ``[B, Q, K]``.

    ``key_chunk_size`` is accepted for API compatibility; the kernel streams
    keys without materialising per-head dots, so no chunking is needed.
    ``causal_offset`` defaults to ``K - Q`` (the last query sees every key).
    """

    del key_chunk_size
    if queries.ndim != 4 or weights.shape != queries.shape[:-1]:
        raise ValueError("queries must be [batch,query,heads,dim]")
    if keys.ndim != 3 or keys.shape[0] != queries.shape[0]:
        raise ValueError("keys must be [batch,key,dim]")
    batch, num_queries, heads, dim = queries.shape
    length = keys.shape[1]
    if heads != HEADS or dim != HEAD_DIM or keys.shape[2] != HEAD_DIM:
        raise ValueError("expected 64 heads x 128 dims")
    if not (queries.is_cuda and weights.is_cuda and keys.is_cuda):
        raise ValueError("HIP kernels require GPU tensors")
    if queries.dtype not in (torch.float16, torch.bfloat16):
        raise ValueError("queries must be FP16/BF16")
    fp8 = keys.dtype == torch.float8_e4m3fn
    if fp8:
        if queries.dtype != torch.bfloat16:
            raise ValueError("fp8 keys are scored against BF16 queries")
        if key_scales is None or key_scales.shape != (batch, (length + 127) // 128):
            raise ValueError("fp8 keys need key_scales [batch, ceil(keys/128)]")
        key_scales = key_scales.to(device=keys.device, dtype=torch.float32).contiguous()
    elif keys.dtype != queries.dtype:
        raise ValueError("queries and keys must share FP16/BF16 dtype")
    if length == 0 or num_queries == 0 or batch == 0:
        return torch.empty((batch, num_queries, length), device=keys.device, dtype=torch.float32)
    queries = queries.contiguous()
    keys = keys.contiguous()
    weights = weights.to(torch.float32).contiguous()
    out = torch.empty((batch, num_queries, length), device=keys.device, dtype=torch.float32)
    offset = -1
    if causal:
        offset = length - num_queries if causal_offset is None else int(causal_offset)
        if offset < 0:
            raise ValueError("causal_offset must be non-negative")
    _lib.call(
        "dsa_score_queries",
        _lib.ptr(queries), HEADS * HEAD_DIM, _lib.ptr(weights), HEADS, None, 0, HEADS,
        _lib.ptr(keys), length, num_queries, _lib.ptr(key_scales), (length + 127) // 128,
        _lib.ptr(out), length, batch * num_queries, length, offset,
        _lib.dtype_code(keys.dtype), _lib.stream_of(keys),
    )
    return out


def score_encoded_topk(
    queries: torch.Tensor,
    weights: torch.Tensor,
    keys: torch.Tensor,
    k: int,
    *,
    causal: bool = False,
    causal_offset: int | None = None,
    return_values: bool = False,
):
    """``score_encoded`` (reference sidecar.py:89-107) and every query's exact
    top-k of its visible keys (``stable_topk``, metrics.py:9-22, in ascending
    index order) in one launch (``dsa_score_queries_topk``).

    Returns ``(scores [B, Q, K] fp32, indices [B, Q, k] int64)``, plus the
    selected values ``[B, Q, k]`` with ``return_values``.  A query with fewer
    than ``k`` visible keys returns all of them, padded with -1 (values -inf).
    Needs fp16/bf16 queries and keys, at least 4 queries per key set and at
    most 4096 keys.
    """

    if queries.ndim != 4 or weights.shape != queries.shape[:-1]:
        raise ValueError("queries must be [batch,query,heads,dim]")
    if keys.ndim != 3 or keys.shape[0] != queries.shape[0]:
        raise ValueError("keys must be [batch,key,dim]")
    batch, num_queries, heads, dim = queries.shape
    length = keys.shape[1]
    if heads != HEADS or dim != HEAD_DIM or keys.shape[2] != HEAD_DIM:
        raise ValueError("expected 64 heads x 128 dims")
    if not (queries.is_cuda and weights.is_cuda and keys.is_cuda):
        raise ValueError("HIP kernels require GPU tensors")
    if queries.dtype not in (torch.float16, torch.bfloat16) or keys.dtype != queries.dtype:
        raise ValueError("queries and keys must share FP16/BF16 dtype")
    if k <= 0:
        raise ValueError("k must be positive")
    if not 1 <= length <= 4096:
        raise ValueError("the fused top-k takes 1..4096 keys per key set")
    if num_queries < 4:
        raise ValueError("the fused top-k takes at least 4 queries per key set")
    offset = -1
    if causal:
        offset = length - num_queries if causal_offset is None else int(causal_offset)
        if offset < 0:
            raise ValueError("causal_offset must be non-negative")
    queries = queries.contiguous()
    keys = keys.contiguous()
    weights = weights.to(torch.float32).contiguous()
    scores = torch.empty((batch, num_queries, length), device=keys.device, dtype=torch.float32)
    indices = torch.empty((batch, num_queries, k), device=keys.device, dtype=torch.int64)
    values = torch.empty((batch, num_queries, k), device=keys.device, dtype=torch.float32) if return_values else None
    _lib.call(
        "dsa_score_queries_topk",
        _lib.ptr(queries), HEADS * HEAD_DIM, _lib.ptr(weights), HEADS, _lib.ptr(keys), length, num_queries,
        _lib.ptr(scores), length, batch * num_queries, length, offset, _lib.dtype_code(keys.dtype), int(k),
        _lib.ptr(indices), _lib.ptr(values), int(k), _lib.stream_of(keys),
    )
    if return_values:
        return scores, indices, values
    return scores, indices


def _row_dtype(t: torch.Tensor) -> int:
    try:
        return _ROW_DTYPES[t.dtype]
    except KeyError:
        raise ValueError("sidecar rows must be float32 or bfloat16") from None


def _token_positions(positions, shape, device) -> torch.Tensor:
    pos = torch.as_tensor(positions, device=device)
    if pos.shape != shape:
        pos = pos.expand(shape)
    return pos.to(torch.int64).contiguous().reshape(-1)


def _hidden_rows(hidden: torch.Tensor, tokens: int, kdim: int) -> torch.Tensor:
    """hidden as ``[tokens, kdim]`` rows the projection kernels can read: unit
    stride inside a row, rows 16-byte aligned."""

    flat = hidden.reshape(tokens, kdim)
    if flat.stride(-1) != 1 or (tokens > 1 and (flat.stride(0) % 8 or flat.stride(0) < kdim)) or flat.data_ptr() % 16:
        flat = flat.contiguous()
        if flat.data_ptr() % 16:
            flat = flat.clone()
    return flat


def _cache_rows(out, out_rows, tokens: int, dim: int, device) -> torch.Tensor:
    """The checked cache row of every token of ``encode_keys(out=...)``."""

    if out.ndim != 2 or out.shape[1] != dim or not out.is_contiguous():
        raise ValueError("out must be a contiguous [rows, head_dim] key cache")
    if out_rows is None or out_rows.numel() != tokens:
        raise ValueError("out_rows must give one cache row per token")
    # (rows outside the cache are skipped by the kernel: no host sync here)
    return out_rows.to(device=device, dtype=torch.int64).contiguous()


def apply_noninterleaved_rope(x: torch.Tensor, positions: torch.Tensor, *, theta: float = 10_000.0) -> torch.Tensor:
    """Non-interleaved RoPE (reference sidecar.py:10-28) of x ``[..., d]``;
    positions has shape ``x.shape[:-1]`` or ``x.shape[:-2]`` (one position
    per token, shared by its heads)."""

    if x.shape[-1] % 2:
        raise ValueError("RoPE dimension must be even")
    if not x.is_cuda:
        raise ValueError("HIP kernels require GPU tensors")
    dtype = _row_dtype(x)
    d = x.shape[-1]
    pos = torch.as_tensor(positions, device=x.device)
    if tuple(pos.shape) == tuple(x.shape[:-1]):
        heads = 1
        tokens_shape = x.shape[:-1]
    elif x.ndim >= 2 and tuple(pos.shape) == tuple(x.shape[:-2]):
        heads = x.shape[-2]
        tokens_shape = x.shape[:-2]
    else:
        raise ValueError("positions must match x.shape[:-1] or x.shape[:-2]")
    if d > 256:
        raise ValueError("RoPE rows of more than 256 dims are not supported")
    rows = x.contiguous()
    out = torch.empty_like(rows)
    tokens = math.prod(tokens_shape)
    _lib.call("dsa_rope", _lib.ptr(rows), _lib.ptr(out), _lib.ptr(_token_positions(pos, tokens_shape, x.device)),
              tokens, heads, d, d, float(theta), dtype, _lib.stream_of(rows))
    return out


def _split_fp32(tokens: int, kdim: int, features: int) -> bool:
    """Whether bf16 hidden states meet fp32 weights with k split over workgroups (``dsa_project_weights``: partial sums
    and a launch that adds them) or in one launch (``dsa_project_gemm``).  Split unless the one launch's workgroups (64
    features x 16 tokens) run in one round and either k is too short to pay for a second launch or the features alone
    leave no CUs to split k over.  One launch / split, us a call: 64 features 1000 x 256 7.5 / 8.9, 64 x 2048 19.6 / 9.5;
    8192 features 17 x 2048 20.5 / 29.9, 64 x 2048 37.8 / 31.6, 2048 x 2048 1074 / 706.  At k 1024 the split is 12.1 / 9.3
    by itself, but the encoders of an fp32 module wait for the host there, 64 tokens 71 / 78."""

    tiles = -(-features // 64)
    one_round = tiles * -(-tokens // 16) <= 256
    return not (one_round and (kdim <= 1024 or tiles * -(-tokens // 64) >= 128))


class LightningIndexerSidecar(nn.Module):
    """The indexer sidecar (reference sidecar.py:31-121): same constructor,
    parameters and initialisation; the encoders' epilogues run in HIP."""

    def __init__(
        self,
        hidden_size: int = 2048,
        heads: int = 64,
        head_dim: int = 128,
        rope_dim: int = 64,
        rope_theta: float = 10_000.0,
    ) -> None:
        super().__init__()
        if not 0 <= rope_dim <= head_dim or rope_dim % 2:
            raise ValueError("rope_dim must be even and no larger than head_dim")
        self.hidden_size = hidden_size
        self.heads = heads
        self.head_dim = head_dim
        self.rope_dim = rope_dim
        self.rope_theta = rope_theta
        self.wq = nn.Linear(hidden_size, heads * head_dim, bias=False)
        self.wk = nn.Linear(hidden_size, head_dim, bias=False)
        self.k_norm = nn.LayerNorm(head_dim, eps=1e-6)
        self.weights_proj = nn.Linear(hidden_size, heads, bias=False, dtype=torch.float32)
        self.reset_parameters()

    def reset_parameters(self) -> None:
        nn.init.normal_(self.wq.weight, mean=0.0, std=self.hidden_size**-0.5)
        nn.init.normal_(self.wk.weight, mean=0.0, std=self.hidden_size**-0.5)
        nn.init.normal_(self.weights_proj.weight, mean=0.0, std=self.hidden_size**-0.5)

    def _project(self, hidden: torch.Tensor, weight: torch.Tensor, *, fp32: bool = False,
                 scale: float | None = None, positions: torch.Tensor | None = None) -> torch.Tensor:
        """A Linear without bias (sidecar.py:55-58): ``hidden @ weight.T``, in
        the weight's dtype (bf16, or fp32 on ``hidden.float()`` with ``fp32``
        as weights_proj runs), times ``scale`` in fp32 when given.  A decode
        step (at most 16 bf16 tokens) streams the weights in
        ``dsa_project_rows``; larger batches, and fp32 modules, run the MFMA
        GEMM ``dsa_project_gemm``, which with ``positions`` also applies
        encode_queries' RoPE to every 128-dim head (bf16, rope_dim 64).
        Inference only: no autograd graph is kept."""

        kdim = hidden.shape[-1]
        if weight.ndim != 2 or weight.shape[1] != kdim:
            raise ValueError(f"hidden width {kdim} does not match the weight's {tuple(weight.shape)}")
        if not hidden.is_cuda or not weight.is_cuda:
            raise ValueError("HIP kernels require GPU tensors")
        tokens = hidden.numel() // kdim if kdim else 0
        features = weight.shape[0]
        w = weight.detach()
        if fp32 and w.dtype != torch.float32:
            w = w.float()
        if hidden.dtype not in (torch.bfloat16, torch.float32) or w.dtype not in (torch.bfloat16, torch.float32):
            raise ValueError("sidecar projections take bf16 or fp32 hidden states and weights")
        if w.dtype == torch.bfloat16 and hidden.dtype != torch.bfloat16:
            raise ValueError("a bf16 projection takes bf16 hidden states")
        w = w.contiguous()
        out_dtype = torch.float32 if w.dtype == torch.float32 else torch.bfloat16
        lead = hidden.shape[:-1]
        out = torch.empty((tokens, features), device=hidden.device, dtype=out_dtype)
        if tokens == 0:
            return out.reshape(*lead, features)
        flat = hidden.reshape(tokens, kdim)
        if flat.stride(-1) != 1 or flat.stride(0) % 8 or flat.data_ptr() % 16:
            flat = flat.contiguous()
        stream = _lib.stream_of(flat)
        decode = (tokens <= 16 and hidden.dtype == torch.bfloat16 and kdim % 32 == 0 and scale is None
                  and positions is None and (w.dtype == torch.float32 or features % 16 == 0))
        if decode:
            _lib.call("dsa_project_rows", _lib.ptr(flat), flat.stride(0), tokens, _lib.ptr(w),
                      _lib.DTYPE_F32 if w.dtype == torch.float32 else _lib.DTYPE_BF16, features, kdim, _lib.ptr(out),
                      features, stream)
            return out.reshape(*lead, features)
        if kdim % 8 or features % 4:
            raise ValueError("sidecar projections need a hidden width that is a multiple of 8 and a multiple of "
                             "4 output features")
        if (w.dtype == torch.float32 and hidden.dtype == torch.bfloat16 and positions is None
                and _split_fp32(tokens, kdim, features)):
            need = int(_lib.query("dsa_project_weights_workspace_bytes", tokens, kdim, features))
            ws = torch.empty(need, device=hidden.device, dtype=torch.uint8)
            _lib.call("dsa_project_weights", _lib.ptr(flat), flat.stride(0), tokens, kdim, _lib.ptr(w), features,
                      float(1.0 if scale is None else scale), _lib.ptr(out), _lib.ptr(ws), need, stream)
            return out.reshape(*lead, features)
        pos = None
        ws = None
        need = 0
        if positions is not None:
            pos = _token_positions(positions, lead, hidden.device)
            need = int(_lib.query("dsa_project_gemm_workspace_bytes", tokens))
            ws = _lib.workspace("rope_table", hidden.device, stream, need, zeroed=False)
        _lib.call("dsa_project_gemm", _lib.ptr(flat), _row_dtype(flat), flat.stride(0), tokens, kdim, _lib.ptr(w),
                  _row_dtype(w), features, _lib.ptr(out), features, float(1.0 if scale is None else scale),
                  _lib.ptr(pos), float(self.rope_theta), _lib.ptr(ws), need, stream)
        return out.reshape(*lead, features)

    def _project_pair(self, hidden: torch.Tensor, weight: torch.Tensor, weight_f32: torch.Tensor):
        """``(hidden @ weight.T, hidden.float() @ weight_f32.T)`` in one
        launch (``dsa_project_rows_pair``) for a decode step that fits the
        projection kernel, else ``None``; identical to two :meth:`_project`
        calls."""

        tokens = hidden.numel() // hidden.shape[-1] if hidden.shape[-1] else 0
        kdim = hidden.shape[-1]
        if not (hidden.is_cuda and 0 < tokens <= 16 and hidden.dtype == torch.bfloat16 and kdim % 32 == 0
                and weight.ndim == 2 and weight.shape[1] == kdim and weight_f32.ndim == 2 and weight_f32.shape[1] == kdim
                and weight.dtype == torch.bfloat16 and weight.shape[0] % 16 == 0 and weight_f32.dtype == torch.float32):
            return None
        flat = hidden.reshape(tokens, kdim)
        if flat.stride(-1) != 1 or flat.stride(0) % 8 or flat.data_ptr() % 16:
            flat = flat.contiguous()
        w = weight.detach().contiguous()
        wf = weight_f32.detach().contiguous()
        out = torch.empty((tokens, w.shape[0]), device=hidden.device, dtype=torch.bfloat16)
        out_f = torch.empty((tokens, wf.shape[0]), device=hidden.device, dtype=torch.float32)
        _lib.call("dsa_project_rows_pair", _lib.ptr(flat), flat.stride(0), tokens, kdim, _lib.ptr(w), w.shape[0],
                  _lib.ptr(out), w.shape[0], _lib.ptr(wf), wf.shape[0], _lib.ptr(out_f), wf.shape[0],
                  _lib.stream_of(flat))
        lead = hidden.shape[:-1]
        return out.reshape(*lead, w.shape[0]), out_f.reshape(*lead, wf.shape[0])

    def encode_keys(
        self,
        hidden: torch.Tensor,
        positions: torch.Tensor,
        *,
        out: torch.Tensor | None = None,
        out_rows: torch.Tensor | None = None,
    ) -> torch.Tensor:
        """RoPE(LayerNorm(wk(hidden))) (sidecar.py:74-76) ``[..., head_dim]``.

        With ``out`` (a key cache ``[rows, head_dim]``, fp32 or bf16) and
        ``out_rows`` (int64, one cache row per token), the keys are written
        into the cache rows instead and ``out`` is returned: the decode step's
        append without a separate copy.  A token whose row lies outside the
        cache is not written.  Inference only: no autograd graph is kept.
        """

        if not hidden.is_cuda:
            raise ValueError("HIP kernels require GPU tensors")
        fused = self._encode_keys_rows(hidden, positions, out, out_rows)
        if fused is not None:
            return fused
        proj = self._project(hidden, self.wk.weight)
        tokens_shape = proj.shape[:-1]
        tokens = math.prod(tokens_shape)
        flat = proj.reshape(tokens, self.head_dim).contiguous()
        pos = _token_positions(positions, tokens_shape, hidden.device)
        ln_w = self.k_norm.weight.detach().to(torch.float32).contiguous()
        ln_b = self.k_norm.bias.detach().to(torch.float32).contiguous()
        if out is None:
            result = torch.empty_like(flat)
            rows = None
            target = result
        else:
            rows = _cache_rows(out, out_rows, tokens, self.head_dim, hidden.device)
            target = out
        _lib.call(
            "dsa_encode_keys_epilogue", _lib.ptr(flat), _row_dtype(flat), self.head_dim, _lib.ptr(ln_w),
            _lib.ptr(ln_b), float(self.k_norm.eps), _lib.ptr(pos), self.rope_dim, float(self.rope_theta),
            _lib.ptr(target), _row_dtype(target), self.head_dim, _lib.ptr(rows), target.shape[0], tokens,
            self.head_dim, _lib.stream_of(flat),
        )
        if out is not None:
            return out
        return result.reshape(*tokens_shape, self.head_dim)

    def _encode_keys_rows(self, hidden, positions, out, out_rows) -> torch.Tensor | None:
        """:meth:`encode_keys` of bf16 hidden states with a bf16 wk in one
        library call, which takes the LayerNorm's parameters as they are
        stored; ``None`` where the separate calls are needed."""

        weight, ln_w, ln_b = self.wk.weight, self.k_norm.weight, self.k_norm.bias
        kdim, dim = hidden.shape[-1], self.head_dim
        tokens = hidden.numel() // kdim if kdim else 0
        if (tokens == 0 or hidden.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16
                or weight.shape != (dim, kdim) or kdim % 8 or dim % 4 or ln_w.dtype != ln_b.dtype
                or ln_w.dtype not in _ROW_DTYPES
                or not (weight.is_cuda and weight.is_contiguous() and ln_w.is_contiguous() and ln_b.is_contiguous())):
            return None
        lead = hidden.shape[:-1]
        pos = _token_positions(positions, lead, hidden.device)
        if out is None:
            target, rows = torch.empty((*lead, dim), device=hidden.device, dtype=torch.bfloat16), None
            limit = tokens
        else:
            target, rows = out, _cache_rows(out, out_rows, tokens, dim, hidden.device)
            limit = out.shape[0]
        flat = _hidden_rows(hidden, tokens, kdim)
        need = int(_lib.query("dsa_encode_keys_workspace_bytes", tokens, kdim, dim))
        ws = torch.empty(need, device=hidden.device, dtype=torch.uint8)
        stride = flat.stride(0) if tokens > 1 else kdim
        _lib.call("dsa_encode_keys_rows", flat.data_ptr(), stride, tokens, kdim, weight.data_ptr(), dim,
                  ws.data_ptr(), need, ln_w.data_ptr(), ln_b.data_ptr(), _ROW_DTYPES[ln_w.dtype], self.k_norm.eps,
                  pos.data_ptr(), self.rope_dim, self.rope_theta, target.data_ptr(), _row_dtype(target), dim,
                  _lib.ptr(rows), limit, _lib.stream_of(flat))
        return target

    def _encode_queries_rows(self, hidden, positions, scale) -> tuple[torch.Tensor, torch.Tensor] | None:
        """:meth:`encode_queries` of a decode step in one launch
        (``dsa_encode_queries_rows``), identical to the separate calls;
        ``None`` where those are needed."""

        wq, wp = self.wq.weight, self.weights_proj.weight
        kdim = hidden.shape[-1]
        tokens = hidden.numel() // kdim if kdim else 0
        if (not 0 < tokens <= 16 or kdim % 32 or hidden.dtype != torch.bfloat16 or wq.dtype != torch.bfloat16
                or wp.dtype != torch.float32 or self.head_dim != HEAD_DIM or self.rope_dim != 64
                or wq.shape != (self.heads * HEAD_DIM, kdim) or wp.shape != (self.heads, kdim)
                or not (wq.is_cuda and wp.is_cuda and wq.is_contiguous() and wp.is_contiguous())):
            return None
        lead = hidden.shape[:-1]
        pos = _token_positions(positions, lead, hidden.device)
        flat = _hidden_rows(hidden, tokens, kdim)
        queries = torch.empty((*lead, self.heads, HEAD_DIM), device=hidden.device, dtype=torch.bfloat16)
        weights = torch.empty((*lead, self.heads), device=hidden.device, dtype=torch.float32)
        stride = flat.stride(0) if tokens > 1 else kdim
        _lib.call("dsa_encode_queries_rows", flat.data_ptr(), stride, tokens, kdim, wq.data_ptr(), self.heads,
                  wp.data_ptr(), pos.data_ptr(), self.rope_theta, scale, queries.data_ptr(), weights.data_ptr(),
                  _lib.stream_of(flat))
        return queries, weights

    def _encode_queries_gemm(self, hidden, positions, scale, tokens) -> tuple[torch.Tensor, torch.Tensor] | None:
        """:meth:`encode_queries` of a batch of bf16 tokens in one library
        call (``dsa_encode_queries_gemm``); ``None`` where the separate calls
        are needed."""

        wq, wp = self.wq.weight, self.weights_proj.weight
        kdim = hidden.shape[-1]
        if (wp.dtype != torch.float32 or self.heads % 4 or wq.shape != (self.heads * HEAD_DIM, kdim)
                or wp.shape != (self.heads, kdim)
                or not (wq.is_cuda and wp.is_cuda and wq.is_contiguous() and wp.is_contiguous())):
            return None
        lead = hidden.shape[:-1]
        pos = _token_positions(positions, lead, hidden.device)
        flat = _hidden_rows(hidden, tokens, kdim)
        queries = torch.empty((*lead, self.heads, HEAD_DIM), device=hidden.device, dtype=torch.bfloat16)
        weights = torch.empty((*lead, self.heads), device=hidden.device, dtype=torch.float32)
        need = int(_lib.query("dsa_encode_queries_workspace_bytes", tokens, kdim, self.heads))
        ws = torch.empty(need, device=hidden.device, dtype=torch.uint8)
        _lib.call("dsa_encode_queries_gemm", flat.data_ptr(), flat.stride(0), tokens, kdim, wq.data_ptr(), self.heads,
                  wp.data_ptr(), pos.data_ptr(), self.rope_theta, scale, queries.data_ptr(), weights.data_ptr(),
                  ws.data_ptr(), need, _lib.stream_of(flat))
        return queries, weights

    def encode_queries(self, hidden: torch.Tensor, positions: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
        """(queries ``[..., heads, head_dim]``, weights ``[..., heads]`` fp32)
        (sidecar.py:78-88)."""

        if not hidden.is_cuda:
            raise ValueError("HIP kernels require GPU tensors")
        scale = float((self.heads * self.head_dim) ** -0.5)
        tokens = hidden.numel() // hidden.shape[-1] if hidden.shape[-1] else 0
        if (tokens > 16 and hidden.dtype == torch.bfloat16 and self.wq.weight.dtype == torch.bfloat16
                and self.head_dim == 128 and self.rope_dim == 64 and (self.heads * self.head_dim) % 256 == 0
                and hidden.shape[-1] % 8 == 0):
            # The RoPE of every head in the wq GEMM's output stage and the
            # head-weight scale in weights_proj's: no epilogue pass.
            fused = self._encode_queries_gemm(hidden, positions, scale, tokens)
            if fused is not None:
                return fused
            lead = hidden.shape[:-1]
            queries = self._project(hidden, self.wq.weight, positions=positions)
            weights = self._project(hidden, self.weights_proj.weight, fp32=True, scale=scale)
            return queries.reshape(*lead, self.heads, self.head_dim), weights.reshape(*lead, self.heads)
        fused = self._encode_queries_rows(hidden, positions, scale)
        if fused is not None:
            return fused
        pair = self._project_pair(hidden, self.wq.weight, self.weights_proj.weight)
        if pair is None:
            proj = self._project(hidden, self.wq.weight)
            proj_w = self._project(hidden, self.weights_proj.weight, fp32=True)
        else:
            proj, proj_w = pair
        tokens_shape = proj.shape[:-1]
        tokens = math.prod(tokens_shape)
        flat = proj.reshape(tokens, self.heads * self.head_dim).contiguous()
        flat_w = proj_w.reshape(tokens, self.heads).contiguous()
        pos = _token_positions(positions, tokens_shape, hidden.device)
        queries = torch.empty_like(flat)
        weights = torch.empty_like(flat_w)
        _lib.call(
            "dsa_encode_queries_epilogue", _lib.ptr(flat), _lib.ptr(flat_w), _lib.ptr(pos), self.rope_dim,
            float(self.rope_theta), scale, _lib.ptr(queries),
            _lib.ptr(weights), tokens, self.heads, self.head_dim, _row_dtype(flat), _lib.stream_of(flat),
        )
        return (queries.reshape(*tokens_shape, self.heads, self.head_dim), weights.reshape(*tokens_shape, self.heads))

    def score_encoded(
        self,
        queries: torch.Tensor,
        weights: torch.Tensor,
        keys: torch.Tensor,
        *,
        key_chunk_size: int | None = None,
    ) -> torch.Tensor:
        """``[B,Q,H,D] x [B,K,D] -> [B,Q,K]`` (sidecar.py:89-107) on the HIP
        scoring kernel: 64 heads x 128 dims, bf16/fp16 queries (fp32 keys are
        cast to the query dtype, as autocast does in the reference's flow)."""

        if keys.is_floating_point() and keys.dtype == torch.float32 and queries.dtype != torch.float32:
            keys = keys.to(queries.dtype)
        return score_encoded(queries, weights, keys, key_chunk_size=key_chunk_size)

    def forward(
        self,
        query_hidden: torch.Tensor,
        key_hidden: torch.Tensor,
        query_positions: torch.Tensor,
        key_positions: torch.Tensor,
        *,
        key_chunk_size: int | None = None,
    ) -> torch.Tensor:
        queries, weights = self.encode_queries(query_hidden, query_positions)
        keys = self.encode_keys(key_hidden, key_positions)
        return self.score_encoded(queries, weights, keys, key_chunk_size=key_chunk_size)
