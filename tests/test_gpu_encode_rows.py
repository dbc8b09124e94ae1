"""The encoders' single-call paths against the separate entry points they
replace, bit for bit: dsa_encode_queries_rows (one launch for a decode step's
wq with RoPE and weights_proj with its scale) against dsa_project_rows_pair
and dsa_encode_queries_epilogue, and dsa_encode_keys_rows (LayerNorm
parameters read as they are stored) against the projection and
dsa_encode_keys_epilogue.  The separate entry points' parity with the oracle is
test_gpu_sidecar.py's and test_gpu_sidecar_gemm.py's.  Batches of tokens sum wk
over k in another order, so there a projection may fall on the other side of a
bf16 rounding: held to the bound below, and equal almost everywhere.  The wq
GEMM's tiles all add k in the same order and are compared bit for bit.
"""

from __future__ import annotations

import pytest
import torch

from dsa_amd import _lib, sidecar

pytestmark = pytest.mark.gpu


def _stream():
    return torch.cuda.current_stream().cuda_stream


@pytest.mark.parametrize("tokens,kdim,heads,offset", [
    (1, 32, 1, 0),      # one k-step: three quarters of k empty
    (3, 96, 3, 0),      # an odd head count leaves half a weights_proj workgroup idle
    (16, 2048, 64, 0),
    (7, 2080, 64, 1),   # a second round of k, weights_proj 4-byte aligned only
    (15, 4096, 5, 0),
])
def test_queries_equal_separate_calls(device, tokens, kdim, heads, offset) -> None:
    print(f"encode queries rows tokens={tokens} kdim={kdim} heads={heads}", flush=True)
    gen = torch.Generator().manual_seed(7 + kdim)
    hidden = torch.randn(tokens, kdim + 8, generator=gen).to(device, torch.bfloat16)[:, :kdim]
    wq = (torch.randn(heads * 128, kdim, generator=gen) * kdim**-0.5).to(device, torch.bfloat16)
    wp = torch.randn(heads * kdim + offset, generator=gen).to(device)[offset:] * kdim**-0.5
    if offset:
        wp = torch.cat([torch.zeros(offset, device=device), wp])[offset:]
        assert wp.data_ptr() % 16
    positions = torch.randint(0, 40000, (tokens,), generator=gen).to(device)
    scale = float((heads * 128) ** -0.5)
    q = torch.empty(tokens, heads, 128, device=device, dtype=torch.bfloat16)
    w = torch.empty(tokens, heads, device=device)
    _lib.call("dsa_encode_queries_rows", hidden.data_ptr(), hidden.stride(0), tokens, kdim, wq.data_ptr(), heads,
              wp.data_ptr(), positions.data_ptr(), 10000.0, scale, q.data_ptr(), w.data_ptr(), _stream())
    pq, pw = torch.empty_like(q), torch.empty_like(w)
    _lib.call("dsa_project_rows_pair", hidden.data_ptr(), hidden.stride(0), tokens, kdim, wq.data_ptr(), heads * 128,
              pq.data_ptr(), heads * 128, wp.data_ptr(), heads, pw.data_ptr(), heads, _stream())
    want_q, want_w = torch.empty_like(q), torch.empty_like(w)
    _lib.call("dsa_encode_queries_epilogue", pq.data_ptr(), pw.data_ptr(), positions.data_ptr(), 64, 10000.0, scale,
              want_q.data_ptr(), want_w.data_ptr(), tokens, heads, 128, _lib.DTYPE_BF16, _stream())
    assert torch.equal(q.view(torch.int16), want_q.view(torch.int16))
    assert torch.equal(w, want_w)


@pytest.mark.parametrize("tokens,hidden_size,norm_dtype,cached", [
    (1, 256, torch.bfloat16, True),
    (16, 2048, torch.float32, False),
    (13, 2048, torch.bfloat16, True),
    (17, 64, torch.bfloat16, True),    # batches: one stage of k
    (40, 264, torch.bfloat16, True),   # a k tail
    (65, 2048, torch.float32, False),  # a second token tile of one token
    (300, 1096, torch.bfloat16, True),
])
def test_keys_equal_separate_calls(device, tokens, hidden_size, norm_dtype, cached) -> None:
    print(f"encode keys rows tokens={tokens} hidden={hidden_size} norm={norm_dtype}", flush=True)
    gen = torch.Generator().manual_seed(11 + tokens)
    torch.manual_seed(11 + tokens)  # the module's weights
    module = sidecar.LightningIndexerSidecar(hidden_size=hidden_size).to(device=device, dtype=torch.bfloat16).eval()
    module.k_norm.to(norm_dtype)
    with torch.no_grad():
        module.k_norm.weight.copy_(1 + 0.1 * torch.randn(128, generator=gen))
        module.k_norm.bias.copy_(0.1 * torch.randn(128, generator=gen))
    hidden = torch.randn(tokens, hidden_size, generator=gen).to(device, torch.bfloat16)
    positions = torch.randint(0, 40000, (tokens,), generator=gen).to(device)
    rows = torch.randperm(512, generator=gen)[:tokens].to(device)
    rows[-1] = 512  # outside the cache: not written
    cache = torch.zeros(512, 128, device=device, dtype=torch.bfloat16)
    got = module.encode_keys(hidden, positions, out=cache if cached else None, out_rows=rows if cached else None)
    proj = module._project(hidden, module.wk.weight)
    want = torch.zeros_like(cache) if cached else torch.empty(tokens, 128, device=device, dtype=torch.bfloat16)
    ln_w, ln_b = module.k_norm.weight.detach().float(), module.k_norm.bias.detach().float()
    _lib.call("dsa_encode_keys_epilogue", proj.data_ptr(), _lib.DTYPE_BF16, 128, ln_w.data_ptr(), ln_b.data_ptr(), 1e-6,
              positions.data_ptr(), 64, 10000.0, want.data_ptr(), _lib.DTYPE_BF16, 128,
              rows.data_ptr() if cached else None, want.shape[0], tokens, 128, _stream())
    if tokens <= 16:
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
        return
    # Fewer than one projection in fifty falls on the other side of a rounding,
    # one bf16 step (2^-7 of it) away; take 16 of a row's 128 as the most.  Such a
    # row's mean moves by at most 16/128 2^-7 M, M its largest projection, and its
    # variance by 16/128 2 (2 M) 2^-7 M, so its 1 / deviation by 2^-9 M^2 / variance
    # of itself.  (A bias that cancels a projection leaves a key far smaller than
    # the step.)  Then at most four more roundings (2^-9 each, on either side) of
    # values no larger than the rotated pair: below 2^-6 of it.
    assert (got != want).float().mean() < 0.02
    x = proj.double()
    largest = x.abs().amax(dim=1, keepdim=True)
    var = x.var(dim=1, unbiased=False, keepdim=True) + 1e-6
    scaled = ln_w.double().abs() / var.sqrt()
    step = scaled * (2.0**-7 * x.abs() + 2.0**-10 * largest)
    step = step + scaled * (x - x.mean(dim=1, keepdim=True)).abs() * 2.0**-9 * largest**2 / var
    rotated = step[:, :32] + step[:, 32:64]
    step = torch.cat((rotated, rotated, step[:, 64:]), dim=1)
    if cached:
        inside = rows < 512
        step = torch.zeros(512, 128, device=device, dtype=torch.float64).index_copy_(0, rows[inside], step[inside])
    wide = want.double()
    pair = wide[..., :32].hypot(wide[..., 32:64])
    size = torch.cat((pair, pair, wide[..., 64:].abs()), dim=-1)
    assert ((got.double() - wide).abs() <= 2.0**-6 * size + step).all()


@pytest.mark.parametrize("tokens", [16, 17, 300])
def test_key_rows_off_an_8_byte_boundary(device, tokens) -> None:
    # A cache view that starts two elements into its storage, and row strides of
    # 130 (even, not whole 8-byte steps) and 129 (odd: rejected for any batch).
    print(f"encode keys misaligned rows tokens={tokens}", flush=True)
    gen = torch.Generator().manual_seed(23 + tokens)
    module = sidecar.LightningIndexerSidecar(hidden_size=256).to(device=device, dtype=torch.bfloat16).eval()
    hidden = torch.randn(tokens, 256, generator=gen).to(device, torch.bfloat16)
    positions = torch.randint(0, 40000, (tokens,), generator=gen).to(device)
    rows = torch.randperm(400, generator=gen)[:tokens].to(device)
    store = torch.zeros(400 * 128 + 2, device=device, dtype=torch.bfloat16)
    view = store[2:].view(400, 128)
    module.encode_keys(hidden, positions, out=view, out_rows=rows)
    # The separate calls' rows, which store two elements at a time.
    proj = module._project(hidden, module.wk.weight)
    ln_w, ln_b = module.k_norm.weight.detach().float(), module.k_norm.bias.detach().float()
    want = torch.zeros(400, 128, device=device, dtype=torch.bfloat16)
    _lib.call("dsa_encode_keys_epilogue", proj.data_ptr(), _lib.DTYPE_BF16, 128, ln_w.data_ptr(), ln_b.data_ptr(), 1e-6,
              positions.data_ptr(), 64, 10000.0, want.data_ptr(), _lib.DTYPE_BF16, 128, rows.data_ptr(), 400, tokens, 128,
              _stream())
    assert torch.equal(view.view(torch.int16), want.view(torch.int16))
    assert (store[:2] == 0).all()

    need = int(_lib.query("dsa_encode_keys_workspace_bytes", tokens, 256, 128))
    ws = torch.empty(need, device=device, dtype=torch.uint8)

    def strided(stride):
        out = torch.zeros(400 * stride, device=device, dtype=torch.bfloat16)
        _lib.call("dsa_encode_keys_rows", hidden.data_ptr(), 256, tokens, 256, module.wk.weight.data_ptr(), 128,
                  ws.data_ptr(), need, module.k_norm.weight.data_ptr(), module.k_norm.bias.data_ptr(), _lib.DTYPE_BF16,
                  1e-6, positions.data_ptr(), 64, 10000.0, out.data_ptr(), _lib.DTYPE_BF16, stride, rows.data_ptr(), 400,
                  _stream())
        return out.view(400, stride)

    got = strided(130)
    assert torch.equal(got[:, :128].contiguous().view(torch.int16), want.view(torch.int16))
    assert (got[:, 128:] == 0).all()
    with pytest.raises(RuntimeError, match="even"):
        strided(129)


@pytest.mark.parametrize("kdim,strided", [(64, False), (136, False), (192, True), (2048, False)])
def test_wq_tiles_agree(device, kdim, strided) -> None:
    # 1100 tokens x 8192 features: 160 wide tiles (kdim a multiple of 64, one to
    # 32 stages, a 76-token tail); slices of 400, 200 and 100 tokens take the
    # 128-, 64- and 32-token tiles.  One slice is held to the float64 product.
    print(f"wq tiles kdim={kdim}", flush=True)
    gen = torch.Generator().manual_seed(3 + kdim)
    module = sidecar.LightningIndexerSidecar(hidden_size=kdim).to(device=device, dtype=torch.bfloat16).eval()
    hidden = torch.randn(1100, kdim + (8 if strided else 0), generator=gen).to(device, torch.bfloat16)[:, :kdim]
    positions = torch.randint(0, 40000, (1100,), generator=gen).to(device)
    whole = module._project(hidden, module.wq.weight)
    rotated = module._project(hidden, module.wq.weight, positions=positions)
    cuts = [0, 400, 600, 700, 1100]
    for a, b in zip(cuts, cuts[1:]):
        assert torch.equal(whole[a:b], module._project(hidden[a:b], module.wq.weight)), (a, b)
        assert torch.equal(rotated[a:b], module._project(hidden[a:b], module.wq.weight, positions=positions[a:b])), (a, b)
    ref = hidden[-80:].double() @ module.wq.weight.double().t()
    scale = hidden[-80:].double().abs() @ module.wq.weight.double().abs().t()
    # one rounding to bf16 (2^-9), fp32 sums of kdim products below 2^-20 of their magnitudes
    assert ((whole[-80:].double() - ref).abs() <= 2.0**-8 * ref.abs() + 2.0**-20 * scale).all()


@pytest.mark.parametrize("tokens", [1791, 1793, 2048])
def test_wq_tiles_agree_off_64(device, tokens) -> None:
    # kdim 136: 224 and 256 tiles of 256 x 256 on eight waves, ragged and whole;
    # slices of 400 tokens take the 128-token tiles.
    print(f"wq 256-token tiles tokens={tokens}", flush=True)
    gen = torch.Generator().manual_seed(tokens)
    module = sidecar.LightningIndexerSidecar(hidden_size=136).to(device=device, dtype=torch.bfloat16).eval()
    hidden = torch.randn(tokens, 136, generator=gen).to(device, torch.bfloat16)
    positions = torch.randint(0, 40000, (tokens,), generator=gen).to(device)
    whole = module._project(hidden, module.wq.weight)
    rotated = module._project(hidden, module.wq.weight, positions=positions)
    for a in range(0, tokens, 400):
        b = min(tokens, a + 400)
        assert torch.equal(whole[a:b], module._project(hidden[a:b], module.wq.weight)), a
        assert torch.equal(rotated[a:b], module._project(hidden[a:b], module.wq.weight, positions=positions[a:b])), a


def test_partial_sums_past_one_slice(device) -> None:
    # 1100 tokens x 8192 fp32 features in three splits of k: 96 KiB of partial
    # sums a token, so two slices; 131089 keys in one split: two slices as well.
    gen = torch.Generator().manual_seed(41)
    tokens, kdim, features = 1100, 1032, 8192
    print(f"project weights slices tokens={tokens} kdim={kdim} features={features}", flush=True)
    hidden = torch.randn(tokens, kdim, generator=gen).to(device, torch.bfloat16)
    weight = (torch.randn(features, kdim, generator=gen) * kdim**-0.5).to(device)
    need = int(_lib.query("dsa_project_weights_workspace_bytes", tokens, kdim, features))
    assert need <= 64 << 20
    ws = torch.empty(need, device=device, dtype=torch.uint8)
    out = torch.empty(tokens, features, device=device)
    _lib.call("dsa_project_weights", hidden.data_ptr(), kdim, tokens, kdim, weight.data_ptr(), features, 0.5,
              out.data_ptr(), ws.data_ptr(), need, _stream())
    ref = 0.5 * (hidden.double() @ weight.double().t())
    size = 0.5 * (hidden.double().abs() @ weight.double().abs().t())
    assert ((out.double() - ref).abs() <= 2.0**-20 * size).all()

    tokens = 131089
    print(f"encode keys slices tokens={tokens}", flush=True)
    module = sidecar.LightningIndexerSidecar(hidden_size=64, heads=2).to(device=device, dtype=torch.bfloat16).eval()
    hidden = torch.randn(tokens, 64, generator=gen).to(device, torch.bfloat16)
    positions = torch.arange(tokens, device=device)
    whole = module.encode_keys(hidden, positions)
    rows = torch.randperm(tokens, generator=gen).to(device)
    cache = module.encode_keys(hidden, positions, out=torch.zeros_like(whole), out_rows=rows)
    assert torch.equal(cache[rows].view(torch.int16), whole.view(torch.int16))
    for a, b in ((0, 65536), (65536, tokens)):
        part = module.encode_keys(hidden[a:b], positions[a:b])
        assert torch.equal(whole[a:b].view(torch.int16), part.view(torch.int16)), a


def test_fp32_module_keeps_partial_sums_small(device) -> None:
    # wq of an fp32 module on bf16 hidden states, 2048 x 8192 outputs (64 MiB):
    # beyond the projections, the rotated queries and the two weight arrays the
    # call takes at most the 64 MiB of partial sums.
    print("fp32 module peak memory", flush=True)
    module = sidecar.LightningIndexerSidecar(hidden_size=2048).to(device).eval()
    hidden = torch.randn(2048, 2048, generator=torch.Generator().manual_seed(5)).to(device, torch.bfloat16)
    positions = torch.arange(2048, device=device)
    module.encode_queries(hidden[:64], positions[:64])
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    queries, weights = module.encode_queries(hidden, positions)
    torch.cuda.synchronize()
    peak = torch.cuda.max_memory_allocated() - before
    own = 2 * (queries.numel() + weights.numel()) * 4
    print(f"  peak {peak / 2**20:.0f} MiB, of it results and projections {own / 2**20:.0f} MiB", flush=True)
    assert peak <= own + (64 << 20) + (1 << 20)


def _f32_products(hidden, weight):
    """The product in float64, and a bound on any fp32 summation of it: 2^-20 of the sum of |h w| (under 2^12 terms, each
    rounded twice at most along a tree of partial sums)."""

    h, w = hidden.double(), weight.double()
    return h @ w.t(), 2.0**-20 * (h.abs() @ w.abs().t())


@pytest.mark.parametrize("kdim", [72, 264, 1096])  # last stage of 8 k; a last split of 8; a last stage of 8 and a short split
@pytest.mark.parametrize("tokens,features", [(17, 4), (65, 68), (64, 64)])  # a token and a feature past whole tiles
def test_fp32_weights_on_bf16_rows_with_tails(device, tokens, features, kdim) -> None:
    print(f"fp32 weights tokens={tokens} features={features} kdim={kdim}", flush=True)
    gen = torch.Generator().manual_seed(tokens + kdim)
    wide = torch.full((tokens, kdim + 24), 1e30, dtype=torch.bfloat16)  # past a row: never read into the sums
    wide[:, :kdim] = torch.randn(tokens, kdim, generator=gen)
    hidden = wide.to(device)[:, :kdim]
    weight = (torch.randn(features, kdim, generator=gen) * kdim**-0.5).to(device)
    ref, bound = _f32_products(hidden, weight)
    need = int(_lib.query("dsa_project_weights_workspace_bytes", tokens, kdim, features))
    ws = torch.empty(need, device=device, dtype=torch.uint8)
    split, whole = torch.empty(tokens, features, device=device), torch.empty(tokens, features, device=device)
    _lib.call("dsa_project_weights", hidden.data_ptr(), hidden.stride(0), tokens, kdim, weight.data_ptr(), features, 1.0,
              split.data_ptr(), ws.data_ptr(), need, _stream())
    _lib.call("dsa_project_gemm", hidden.data_ptr(), _lib.DTYPE_BF16, hidden.stride(0), tokens, kdim, weight.data_ptr(),
              _lib.DTYPE_F32, features, whole.data_ptr(), features, 1.0, None, 0.0, None, 0, _stream())
    assert ((split.double() - ref).abs() <= bound).all()
    assert ((whole.double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("tokens,kdim,heads", [(17, 72, 4), (65, 264, 68), (64, 1096, 4), (300, 128, 68)])
def test_query_batches_of_other_head_counts(device, tokens, kdim, heads) -> None:
    # The one-call encoder against the plain projection and its epilogue (bit
    # for bit, as every wq tile adds k in the same order), that projection
    # against float64 (half a bf16 ulp, 2^-8 of the value, and the sum's error),
    # and the head weights with their scale, one more rounding.
    print(f"encode queries gemm tokens={tokens} kdim={kdim} heads={heads}", flush=True)
    gen = torch.Generator().manual_seed(tokens + heads)
    hidden = torch.randn(tokens, kdim + 16, generator=gen).to(device, torch.bfloat16)[:, :kdim]
    wq = (torch.randn(heads * 128, kdim, generator=gen) * kdim**-0.5).to(device, torch.bfloat16)
    wp = (torch.randn(heads, kdim, generator=gen) * kdim**-0.5).to(device)
    positions = torch.randint(0, 40000, (tokens,), generator=gen).to(device)
    scale = float((heads * 128) ** -0.5)
    q = torch.empty(tokens, heads, 128, device=device, dtype=torch.bfloat16)
    w = torch.empty(tokens, heads, device=device)
    need = int(_lib.query("dsa_encode_queries_workspace_bytes", tokens, kdim, heads))
    ws = torch.empty(need, device=device, dtype=torch.uint8)
    _lib.call("dsa_encode_queries_gemm", hidden.data_ptr(), hidden.stride(0), tokens, kdim, wq.data_ptr(), heads,
              wp.data_ptr(), positions.data_ptr(), 10000.0, scale, q.data_ptr(), w.data_ptr(), ws.data_ptr(), need,
              _stream())
    plain = torch.empty(tokens, heads * 128, device=device, dtype=torch.bfloat16)
    _lib.call("dsa_project_gemm", hidden.data_ptr(), _lib.DTYPE_BF16, hidden.stride(0), tokens, kdim, wq.data_ptr(),
              _lib.DTYPE_BF16, heads * 128, plain.data_ptr(), heads * 128, 1.0, None, 0.0, None, 0, _stream())
    want = torch.empty_like(q)
    unused = torch.empty_like(w)
    _lib.call("dsa_encode_queries_epilogue", plain.data_ptr(), w.data_ptr(), positions.data_ptr(), 64, 10000.0, scale,
              want.data_ptr(), unused.data_ptr(), tokens, heads, 128, _lib.DTYPE_BF16, _stream())
    assert torch.equal(q.view(torch.int16), want.view(torch.int16))
    ref, bound = _f32_products(hidden, wq)
    assert ((plain.double() - ref).abs() <= 2.0**-8 * ref.abs() + 2 * bound).all()
    ref, bound = _f32_products(hidden, wp)
    assert ((w.double() - scale * ref).abs() <= scale * (bound + 2.0**-23 * ref.abs())).all()


@pytest.mark.parametrize("tokens,features,kdim,split", [
    (17, 8192, 1032, False),   # 128 feature tiles, one round of the unsplit product
    (33, 8192, 520, True),     # a second round
    (256, 1024, 1024, False),  # one round, short k
    (257, 1024, 1024, True),
    (256, 1024, 1032, True),   # one round, k past 1024
])
def test_fp32_weights_split_or_not(device, tokens, features, kdim, split) -> None:
    print(f"fp32 weights dispatch tokens={tokens} features={features} kdim={kdim}", flush=True)
    assert sidecar._split_fp32(tokens, kdim, features) == split
    gen = torch.Generator().manual_seed(tokens + features)
    module = sidecar.LightningIndexerSidecar(hidden_size=kdim)
    hidden = torch.randn(tokens, kdim, generator=gen).to(device, torch.bfloat16)
    weight = (torch.randn(features, kdim, generator=gen) * kdim**-0.5).to(device)
    ref, bound = _f32_products(hidden, weight)
    out = module._project(hidden, weight, fp32=True)
    scaled = module._project(hidden, weight, fp32=True, scale=0.25)
    assert ((out.double() - ref).abs() <= bound).all()
    assert torch.equal(scaled, 0.25 * out)
