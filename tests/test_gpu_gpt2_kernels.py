"""The GPT-2 block kernels (include/tfgfa_gpt2.h) against float64 references of the same
functions, and the modules that use them against their torch operators (needs a GPU, except the
argument checks).

Tolerances.  Values are float32 with float32 sums: a result carries a few roundings of 2^-24
relative to the terms it is made of, so the relative 2-norm error is held to 1e-6 (8 roundings of
2^-23).  bf16 results are rounded once more, to 8 significant bits: half a unit in the last place is at most 2^-8 of the value.
"""
import math

import pytest
import torch

import custom_flash_attn  # noqa: F401
import model_inference as mi
from custom_flash_attn import _C

DEV = "cuda:0"
F32, BF16 = 1e-6, 2.0 ** -8


def _rel(x, ref):
    x, ref = x.double(), ref.double()
    return ((x - ref).norm() / ref.norm()).item()


def _randn(g, *shape):
    return torch.randn(shape, device=DEV, generator=g)


def _norm64(x, scale, shift, eps=1e-5):
    x = x.double()
    y = (x - x.mean(-1, keepdim=True)) / torch.sqrt(x.var(-1, keepdim=True, unbiased=False) + eps)
    return y * scale.double() + shift.double()


def _gelu64(x):
    x = x.double()
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def test_kernel_arguments_are_checked_before_any_hip_call():
    P, F = 0x10000, _C.GPT2_F32
    for kind in (-1, _C.GPT2_PLANES + 1):
        with pytest.raises(RuntimeError, match="dtype"):
            _C.gpt2_layernorm(P, 0, 0, P, P, P, kind, 1, 64, 1e-5, 0)
    with pytest.raises(RuntimeError, match="negative batch|shape|size"):
        _C.gpt2_layernorm(P, 0, 0, P, P, P, F, 1, 6, 1e-5, 0)          # width not a multiple of 4
    with pytest.raises(RuntimeError):
        _C.gpt2_layernorm(P, 0, 0, P, P, P, F, 1, 2052, 1e-5, 0)       # too wide
    with pytest.raises(RuntimeError, match="null"):
        _C.gpt2_layernorm(P, P, 0, P, P, P, F, 1, 64, 1e-5, 0)         # delta without sum
    with pytest.raises(RuntimeError, match="misaligned"):
        _C.gpt2_layernorm(P + 4, 0, 0, P, P, P, F, 1, 64, 1e-5, 0)
    _C.gpt2_layernorm(0, 0, 0, 0, 0, 0, F, 0, 64, 1e-5, 0)             # no rows: nothing to do
    with pytest.raises(RuntimeError, match="misaligned"):
        _C.gpt2_gelu(P + 8, P, 4, 0)
    _C.gpt2_gelu(0, 0, 0, 0)
    with pytest.raises(RuntimeError, match="shape|size"):
        _C.gpt2_cast_bf16([(P, P, 6)], 0)
    with pytest.raises(RuntimeError, match="shape|size"):
        _C.gpt2_cast_bf16([(P, P, 4)] * 11, 0)
    with pytest.raises(RuntimeError, match="misaligned"):
        _C.gpt2_cast_bf16([(P, P + 8, 4)], 0)
    _C.gpt2_cast_bf16([], 0)
    with pytest.raises(RuntimeError, match="shape|size"):
        _C.gpt2_linear_planes(P, P, 0, False, 0, P, P, 1, 4, 6, 32, 0)                        # N not a multiple of 4
    with pytest.raises(RuntimeError, match="shape|size"):
        _C.gpt2_linear_planes(P, P, 0, False, 0, P, P, 1, 4, 8, 48, 0)                        # K not of 32
    with pytest.raises(RuntimeError, match="shape|size"):
        _C.gpt2_linear_planes(P, P, 0, False, 0, P, P, 3, 4, 8, 64, 0)                        # more splits than steps
    with pytest.raises(RuntimeError, match="null"):
        _C.gpt2_linear_planes(P, P, 0, False, 0, P, 0, 2, 4, 8, 64, 0)                        # splits without part
    part = (P, 0, P)
    with pytest.raises(RuntimeError, match="shape|size"):
        _C.gpt2_linear_rows(P, False, 0, 0, 0.0, [part], False, 0, False, 9, 4, 64, 0)       # too many rows
    with pytest.raises(RuntimeError, match="shape|size"):
        _C.gpt2_linear_rows(P, False, P, P, 1e-5, [part], False, 0, False, 8, 4, 2048, 0)    # rows past LDS
    with pytest.raises(RuntimeError, match="shape|size"):
        _C.gpt2_linear_rows(P, False, 0, 0, 0.0, [part] * 4, False, 0, False, 1, 4, 64, 0)
    with pytest.raises(RuntimeError, match="shape|size"):
        _C.gpt2_linear_rows(P, False, 0, 0, 0.0, [part] * 2, False, P, False, 1, 4, 64, 0)   # residual of two parts
    with pytest.raises(RuntimeError, match="dtype"):
        _C.gpt2_linear_rows(P, False, 0, 0, 0.0, [part], False, 0, True, 1, 4, 64, 0)        # bf16 without a norm
    with pytest.raises(RuntimeError, match="misaligned"):
        _C.gpt2_linear_rows(P, False, 0, 0, 0.0, [(P + 4, 0, P)], False, 0, False, 1, 4, 64, 0)


def test_sizes_past_one_launch_are_refused_before_any_hip_call():
    """HIP launches fewer than 2^32 threads: past that the entry points say so, and the modules keep
    their torch operators (sizes of meta tensors only)."""
    from custom_flash_attn import gpt2

    P, big = 0x10000, "launch limits"
    assert gpt2.MAX_NORM_ROWS * 64 < 2 ** 32 <= (gpt2.MAX_NORM_ROWS + 1) * 64
    with pytest.raises(RuntimeError, match=big):
        _C.gpt2_layernorm(P, 0, 0, P, P, P, 0, gpt2.MAX_NORM_ROWS + 1, 4, 1e-5, 0)
    with pytest.raises(RuntimeError, match=big):
        _C.gpt2_gelu(P, P, gpt2.MAX_VALUES + 1, 0)
    with pytest.raises(RuntimeError, match=big):
        _C.gpt2_cast_bf16([(P, P, gpt2.MAX_VALUES), (P, P, 4)], 0)
    for K, norm in ((64, P), (64, 0), (8192, 0)):
        N = 4 * (2 ** 32 // (256 if norm else 512 if K <= 4096 else 1024))
        with pytest.raises(RuntimeError, match=big):
            _C.gpt2_linear_rows(P, False, norm, norm, 0.0, [(P, 0, P)], False, 0, False, 1, N, K, 0)
    norm = mi.LayerNorm({"emb_dim": 32}).to("meta")
    assert norm._native(torch.empty(gpt2.MAX_NORM_ROWS, 32, device="meta"))
    assert not norm._native(torch.empty(gpt2.MAX_NORM_ROWS + 1, 32, device="meta"))
    assert gpt2.rows_fit(1, _C.GPT2_MAX_OUTPUTS, False) and not gpt2.rows_fit(1, _C.GPT2_MAX_OUTPUTS + 4, False)


@pytest.mark.parametrize("d", [4, 28, 32])
def test_many_narrow_rows_stay_with_torch(d):
    """Up to 28 values a row the torch operators take less time than a wave per row from some 37000 rows."""
    norm = mi.LayerNorm({"emb_dim": d}).to("meta")
    assert norm._native(torch.empty(32768, d, device="meta"))
    assert norm._native(torch.empty(300000, d, device="meta")) is (d >= 32)


@pytest.mark.gpu
def test_values_past_one_launch_stay_with_torch(monkeypatch):
    from custom_flash_attn import gpt2

    x, calls = torch.ones(8, device=DEV), []
    monkeypatch.setattr(gpt2, "gelu", lambda x: (calls.append(1), x)[1])
    mi.GELU()(x)
    assert calls
    monkeypatch.setattr(gpt2, "MAX_VALUES", 7)
    torch.testing.assert_close(mi.GELU()(x), torch.nn.functional.gelu(x, approximate="tanh"))
    assert len(calls) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("rows,d", [(1, 4), (3, 252), (4, 256), (5, 260), (7, 768), (2, 1024), (3, 1028),
                                    (9, 1600), (1, 2048)])
def test_layernorm_matches_float64(rows, d):
    """Widths at the edges of a lane's four values, of a wave's 256 and of the two register sizes;
    one and several rows (a workgroup each); an offset mean, so the variance must be centred."""
    from custom_flash_attn import gpt2

    g = torch.Generator(device=DEV).manual_seed(rows * 10007 + d)
    x, scale, shift = _randn(g, rows, d) * 3 + 100, 1 + _randn(g, d), _randn(g, d)
    delta = (_randn(g, rows, d) * 2).to(torch.bfloat16)
    # The centred values lose log2(100 / 3) bits of x's 24.
    y = gpt2.layernorm(x, scale, shift, 1e-5)
    assert _rel(y, _norm64(x, scale, shift)) <= 40 * F32
    s, y = gpt2.layernorm(x, scale, shift, 1e-5, delta=delta)
    assert torch.equal(s, x + delta)
    assert _rel(y, _norm64(s, scale, shift)) <= 40 * F32
    y = gpt2.layernorm(x, scale, shift, 1e-5, torch.bfloat16)
    assert y.dtype == torch.bfloat16 and _rel(y, _norm64(x, scale, shift)) <= BF16


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 3, 4, 1023, 1024, 1025, 40000])
def test_gelu_matches_float64(n):
    from custom_flash_attn import gpt2

    x = _randn(torch.Generator(device=DEV).manual_seed(n), n) * 3
    assert _rel(gpt2.gelu(x), _gelu64(x)) <= F32
    special = torch.tensor([math.inf, -math.inf, math.nan, 0.0, -0.0, 3e38, -3e38, 1e-40, 50.0, -50.0], device=DEV)
    want = 0.5 * special * (1 + torch.tanh(math.sqrt(2.0 / math.pi) * (special + 0.044715 * torch.pow(special, 3))))
    assert torch.equal(gpt2.gelu(special).nan_to_num(nan=7.0), want.nan_to_num(nan=7.0))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 1, 4), (4, 8, 64), (5, 9, 60), (8, 7, 256), (3, 192, 516), (8, 1600, 1600),
                                   (4, 1024, 4096), (2, 33, 2048), (7, 20, 1028)])
def test_linear_rows_matches_float64(M, N, K):
    """Rows at the edges of the column groups, outputs that do not fill a workgroup, widths that
    end inside a strip or a wave's batch of strips; with and without norm, GELU, residual, bias and
    several weight matrices, in every type.  A dot product's float32 error grows as sqrt(K) in the
    mean; the sums here are split over 128 partial ones, so F32 holds for every K."""
    from custom_flash_attn import gpt2

    g = torch.Generator(device=DEV).manual_seed(M * 1009 + N * 31 + K)
    x = _randn(g, M, 1, K)
    parts = [(_randn(g, N, K) * 0.1, _randn(g, N)), (_randn(g, N, K) * 0.1, None), (_randn(g, N, K) * 0.1, _randn(g, N))]
    res = _randn(g, M, 1, N)
    assert gpt2.rows_fit(M, K, False)

    def lin(x, w, b):
        y = x.double() @ w.double().t().contiguous()
        return y if b is None else y + b.double()

    for xx in (x, x.to(torch.bfloat16)):
        for got, (w, b) in zip(gpt2.linear_rows(xx, parts, torch.float32), parts):
            assert _rel(got, lin(xx, w, b)) <= F32
        got, = gpt2.linear_rows(xx, parts[1:2], torch.float32, residual=res)
        assert _rel(got, lin(xx, *parts[1]) + res.double()) <= F32
    if gpt2.rows_fit(M, K, True):
        scale, shift = 1 + _randn(g, K), _randn(g, K)
        xn = _norm64(x, scale, shift)
        for got, (w, b) in zip(gpt2.linear_rows(x, parts, torch.bfloat16, norm=(scale, shift, 1e-5)), parts):
            assert _rel(got, lin(xn, w, b)) <= BF16
        got, = gpt2.linear_rows(x, parts[:1], torch.float32, norm=(scale, shift, 1e-5))
        assert _rel(got, lin(xn, *parts[0])) <= 2 * F32
        got, = gpt2.linear_rows(x, parts[:1], torch.float32, norm=(scale, shift, 1e-5), gelu=True, residual=res)
        assert _rel(got, _gelu64(lin(xn, *parts[0])) + res.double()) <= 2 * F32
    # Infinities stay where they belong: only their row, and no NaN from the padding.
    xi = x.clone()
    xi[0, 0, 0] = math.inf
    got, = gpt2.linear_rows(xi, parts[1:2], torch.float32)
    assert torch.isinf(got[0]).all() and torch.isfinite(got[1:]).all()


def _to_planes(x):
    out = []
    for _ in range(3):
        t = x.to(torch.bfloat16)
        cut = (x.view(torch.int32) & -65536).view(torch.float32).to(torch.bfloat16)
        out.append(torch.where(x.isfinite() & ~t.isfinite(), cut, t))  # no finite value becomes infinite
        x = x - out[-1].float()
    return torch.stack(out)


def _planes64(p):
    return p.double().sum(0)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 4, 32), (9, 128, 64), (127, 132, 96), (128, 124, 128), (129, 260, 160),
                                   (300, 768, 3072), (65, 3072, 768), (613, 1600, 1600)])
def test_linear_planes_matches_float64(M, N, K):
    """Rows and outputs at the edges of a 128 tile, contractions of one to many steps, one and several
    splits, with GELU planes out, with a residual, without a bias; values over eight orders of
    magnitude.  Planes hold 24 bits: a value comes back exactly.  A product is off by at most 2^-26
    of itself (the three dropped terms), sums are float32, so F32 holds as for the other linears; it must
    also be no further from float64 than torch's float32 linear (x 1.25 for the chance of one draw)."""
    from custom_flash_attn import gpt2

    g = torch.Generator(device=DEV).manual_seed(M * 7 + N * 3 + K)
    scale, shift = 1 + _randn(g, K) * 0.1, _randn(g, K) * torch.exp(_randn(g, K) * 3)
    x = _randn(g, M, K)
    xn = _norm64(x, scale, shift).float()
    xp = _to_planes(xn)
    if K <= gpt2.MAX_NORM_DIM:
        xn = gpt2.layernorm(x, scale, shift, 1e-5)
        xp = gpt2.layernorm(x, scale, shift, 1e-5, planes=True)
        assert torch.equal(xp, _to_planes(xn))
    assert torch.equal(_planes64(xp), xn.double())
    w, b, res = _randn(g, N, K) * 0.05, _randn(g, N), _randn(g, M, N)
    y64 = xn.double() @ w.double().t().contiguous()
    lib = _rel(torch.nn.functional.linear(xn, w, b), y64 + b.double())
    auto = gpt2.planes_splits(M, w)
    assert 1 <= auto <= 8
    for splits in sorted({1, auto, min(3, K // 32), min(8, K // 32)}):
        got = gpt2.linear_planes(xp, w, b, splits, residual=res)
        assert _rel(got, y64 + b.double() + res.double()) <= F32
        got = gpt2.linear_planes(xp, w, b, splits)
        assert _rel(got, y64 + b.double()) <= min(F32, max(1.25 * lib, 2e-7))
        got = gpt2.linear_planes(xp, w, None, splits, gelu=True)
        assert got.shape == (3, M, N) and _rel(_planes64(got), _gelu64(y64)) <= F32


@pytest.mark.gpu
@pytest.mark.parametrize("splits", [1, 3])
def test_linear_planes_passes_infinities_as_float32_does(splits):
    """Infinities, NaN, values that round to infinity as bf16 and products that overflow, in x and in
    the weights, one row or output each: infinite and NaN results where float32's linear has them
    (no sum here overflows depending on its order), the finite ones to F32 of the sum of their terms'
    magnitudes."""
    from custom_flash_attn import gpt2

    top = torch.finfo(torch.float32).max
    g = torch.Generator(device=DEV).manual_seed(11)
    M, N, K = 133, 136, 160
    x, w, b = _randn(g, M, K), _randn(g, N, K) * 0.05, _randn(g, N)
    w[:, 3] = torch.where(torch.arange(N, device=DEV) % 2 == 0, 0.5, -0.25)  # exact in bf16: lower parts zero
    w[5, 3] = 0.0
    x[2, 3], x[3, 3], x[4, 3], x[132, 3] = math.inf, -math.inf, math.nan, math.inf
    x[6, 3], x[7, 3] = top, -top * (1 - 2.0 ** -10)
    x[8, 150], x[8, 151] = math.inf, -math.inf   # the last step, alone and against each other
    x[9, :] = 1e30
    w[7, :] = 1e30                               # products past the float range
    w[20, 77], w[21, 78], w[22, 79] = math.inf, math.nan, top
    x[:, 79] = torch.sign(x[:, 79]) * 0.25
    x64, w64, b64 = x.double().cpu(), w.double().cpu(), b.double().cpu()
    ref = torch.nn.functional.linear(x64, w64, b64)
    terms = torch.nn.functional.linear(x64.abs(), w64.abs(), b64.abs())
    got = gpt2.linear_planes(_to_planes(x), w, b, splits).cpu()
    ref32 = ref.float()                          # float32's range: 1e60 is infinite
    assert torch.equal(got.isnan(), ref32.isnan())
    assert torch.equal(got[ref32.isinf()], ref32[ref32.isinf()])
    fin = ref32.isfinite()
    assert 0 < fin.sum() < fin.numel() and ((got.double() - ref).abs() <= F32 * terms)[fin].all()


@pytest.mark.gpu
@pytest.mark.parametrize("splits", [1, 3])
def test_linear_planes_results_at_the_top_of_the_range(splits):
    """Results within 2^-8 of the largest float, of operands whose first bf16 pieces round up past it:
    finite, and to F32 of the float64 result, as float32 products give them; past the range infinite."""
    from custom_flash_attn import gpt2

    M, N, K = 5, 8, 96
    x, w = torch.zeros(M, K, device=DEV), torch.zeros(N, K, device=DEV)
    x[0, 0], x[1, 0], x[2, 40], x[3, 0], x[4, 95] = 1.9999, -1.9999, 2 - 2.0 ** -20, 2.0, 1.5
    w[1::2, :] = 2.0 ** 127
    w[2, :] = 2.0 ** 127 - 2.0 ** 106
    ref = (x.double() @ w.double().t().contiguous()).float()
    got = gpt2.linear_planes(_to_planes(x), w, None, splits)
    assert ref[0].isfinite().all() and ref[3, 1].isinf() and ref[:3].abs().max() > 3.4e38
    assert torch.equal(got.isfinite(), ref.isfinite()) and not got.isnan().any()
    fin = ref.isfinite()
    assert _rel(got[fin].double() * 2.0 ** -64, ref[fin].double() * 2.0 ** -64) <= F32


@pytest.mark.gpu
def test_planes_hold_the_top_of_the_float_range():
    """A norm's result that is finite but rounds to infinity as bf16 comes back from its planes exactly."""
    from custom_flash_attn import gpt2

    K = 64
    x = torch.where(torch.arange(K, device=DEV) % 2 == 0, 1.0, -1.0).repeat(3, 1)   # its own norm
    shift = torch.zeros(K, device=DEV)
    scale = torch.full((K,), torch.finfo(torch.float32).max, device=DEV) * (1 - torch.arange(K, device=DEV) * 2.0 ** -13)
    y = gpt2.layernorm(x, scale, shift, 1e-9)
    assert y.isfinite().all() and not y.to(torch.bfloat16).isfinite().all()
    assert torch.equal(_planes64(gpt2.layernorm(x, scale, shift, 1e-9, planes=True)), y.double())


@pytest.mark.gpu
def test_cast_rounds_as_torch_does():
    """Arrays from one value group up to several workgroups, in one launch, bit for bit."""
    from custom_flash_attn import gpt2

    g = torch.Generator(device=DEV).manual_seed(5)
    src = [_randn(g, n) for n in (4, 1020, 1024, 1028, 40000, 8, 4, 12, 16, 4)]
    src[1][:6] = torch.tensor([math.inf, -math.inf, math.nan, 3.4e38, 1e-40, -0.0], device=DEV)
    dst = [torch.full((t.numel() + 8,), 7.0, dtype=torch.bfloat16, device=DEV) for t in src]
    gpt2.cast_bf16([(s, d[:s.numel()]) for s, d in zip(src, dst)])
    for s, d in zip(src, dst):
        want = torch.cat((s.to(torch.bfloat16), torch.full((8,), 7.0, dtype=torch.bfloat16, device=DEV)))
        assert torch.equal(d.nan_to_num(nan=9.0), want.nan_to_num(nan=9.0))


@pytest.mark.gpu
@pytest.mark.parametrize("impl", ["hip", "cuda", "triton"])
@pytest.mark.parametrize("emb,heads,bias,dtype", [(256, 4, True, torch.float32), (320, 5, False, torch.bfloat16)])
def test_attention_layer_casts_together(impl, emb, heads, bias, dtype):
    """The layer with its casts in one launch and one GEMM for queries, keys and values against the
    layer with a hook on one linear (autocast's casts, four GEMMs).  The bf16 inputs are the same; a
    different summation order flips bf16 roundings, half a unit (2^-8) at most in each result."""
    torch.manual_seed(emb)
    m = mi.MultiHeadAttention(emb, emb, 128, 0.0, heads, impl, qkv_bias=bias).to(DEV).eval()
    x = _randn(torch.Generator(device=DEV).manual_seed(3), 2, 75, emb).to(dtype)
    with torch.no_grad(), torch.autocast("cuda", torch.bfloat16):
        assert m._cast_together(x)
        got = m(x)
        hook = m.W_key.register_forward_hook(lambda *a: None)
        assert not m._cast_together(x)
        want = m(x)
        hook.remove()
    assert got.dtype == want.dtype == torch.bfloat16 and _rel(got, want) <= BF16
    with torch.no_grad(), torch.autocast("cuda", torch.float16):
        assert not m._cast_together(x)


def _block(emb, heads, **kw):
    cfg = dict(mi.GPT_CONFIG_124M)
    cfg.update({"emb_dim": emb, "n_heads": heads, "context_length": 128, "drop_rate": 0.0, "qkv_bias": True,
                "impl_type": "hip", **kw})
    blk = mi.TransformerBlock(cfg).to(DEV).eval()
    g = torch.Generator(device=DEV).manual_seed(emb)
    with torch.no_grad():
        for p in blk.parameters():
            p.add_(_randn(g, *p.shape) * 0.05)
    return blk, g


@pytest.mark.gpu
@pytest.mark.parametrize("emb,heads,bias", [(256, 4, True), (512, 8, False)])
def test_block_matches_its_torch_operators(emb, heads, bias):
    """The fused block against the same block on its torch operators, which a gradient-requiring
    input selects.  The attention's bf16 results are the difference: 2^-8 of its share of x."""
    blk, g = _block(emb, heads, qkv_bias=bias)
    x = _randn(g, 2, 37, emb)
    with torch.no_grad():
        fused = blk(x)
    assert blk._fused(x) is False  # parameters need a gradient outside no_grad
    hook = blk.norm1.register_forward_hook(lambda m, i, o: None)
    seen = []
    hook2 = blk.norm2.register_forward_hook(lambda m, i, o: seen.append(o.shape))
    with torch.no_grad():
        assert not blk._fused(x)
        hooked = blk(x)
    hook.remove()
    hook2.remove()
    assert seen == [x.shape] and _rel(hooked, fused) <= 1e-3


@pytest.mark.gpu
@pytest.mark.parametrize("rows,split", [(1023, False), (1024, True), (1037, True)])
def test_block_mlp_on_split_float32(rows, split):
    """Either side of the size from which the block's MLP runs on the split-float32 kernel, against the
    general path (a hook on the MLP): the attention is the same, the MLP float32 on both."""
    blk, g = _block(512, 8, context_length=1100)
    x = _randn(g, 1, rows, 512)
    with torch.no_grad():
        assert (blk._mlp_splits(x) is not None) is split
        got = blk(x)
        hook = blk.ff.register_forward_hook(lambda *a: None)
        assert blk._mlp_splits(x) is None
        want = blk(x)
        hook.remove()
    assert _rel(got, want) <= 2 * F32


@pytest.mark.gpu
@pytest.mark.parametrize("rows,max_len", [(1, 40), (8, 40), (9, 40)])
def test_decode_step_matches_the_general_path(rows, max_len):
    """A block's decode step on the few-row kernels (up to 8 rows) against the same step with a
    hook on it, which takes the general path; both append the same cache row.  The two differ by
    the bf16 roundings of autocast: 2^-8 of the attention's share of x."""
    blk, g = _block(256, 4)
    cfg = {"n_heads": 4, "emb_dim": 256, "n_layers": 1}
    out = []
    xs = _randn(g, rows, 21, 256)
    new = xs[:, 20:].contiguous()
    for general in (False, True):
        cache = mi.KVCache(cfg, rows, max_len, DEV)
        hook = blk.ff.register_forward_hook(lambda m, i, o: None) if general else None
        with torch.no_grad():
            blk(xs[:, :20], cache, 0)
            cache.advance(20)
            assert blk._rows_fused(new, cache) is (rows <= 8 and not general)
            out.append((blk(new, cache, 0), cache.k[0].clone(), cache.v[0].clone()))
        if hook is not None:
            hook.remove()
    for a, b in zip(*out):
        assert torch.isfinite(a).all() and _rel(a, b) <= 4e-3


@pytest.mark.gpu
def test_modules_keep_gradients_and_transforms():
    """Where a gradient, a function transform, forward-mode or another type is in play the modules
    run their torch operators."""
    norm, act = mi.LayerNorm({"emb_dim": 64}).to(DEV), mi.GELU()
    g = torch.Generator(device=DEV).manual_seed(1)
    x = _randn(g, 5, 64)
    y = act(norm(x))
    y.sum().backward()
    assert norm.scale.grad is not None and torch.isfinite(norm.scale.grad).all()
    with torch.no_grad():
        ref = act(norm(x))
        torch.testing.assert_close(torch.func.vmap(lambda r: act(norm(r)))(x), ref, rtol=1e-5, atol=1e-5)
        torch.testing.assert_close(act(norm(x.double())), ref.double(), rtol=1e-5, atol=1e-5)
        torch.testing.assert_close(act(norm(x.t().contiguous().t())), ref, rtol=1e-5, atol=1e-5)
        with torch.autograd.forward_ad.dual_level():
            dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
            out = act(dual)
            assert torch.autograd.forward_ad.unpack_dual(out).tangent is not None
    assert norm(torch.empty(0, 64, device=DEV)).shape == (0, 64)


@pytest.mark.parametrize("tokens", [16, 17])
def test_last_logits_are_the_models_last_position(tokens):
    """The logits a generation loop samples from, with the head on the last position only past 32
    rows, against the whole model's (CPU, float32: the same sums in another blocking); a hook on the
    head sees every position."""
    cfg = dict(mi.GPT_CONFIG_124M)
    cfg.update({"emb_dim": 64, "n_layers": 2, "n_heads": 2, "vocab_size": 50, "context_length": 32,
                "drop_rate": 0.0, "impl_type": "manual"})
    torch.manual_seed(0)
    model = mi.GPTModel(cfg).eval()
    idx = torch.randint(0, 50, (2, tokens))
    with torch.no_grad():
        want = model(idx)[:, -1, :]
        got = mi._last_logits(model, idx)
        assert got.shape == want.shape and _rel(got, want) <= F32
        seen = []
        hook = model.out_head.register_forward_hook(lambda m, i, o: seen.append(o.shape[1]))
        assert torch.equal(mi._last_logits(model, idx), want)
        hook.remove()
    assert seen == [tokens]


def test_compiled_modules_are_called():
    """A module that was compiled in place runs its compiled form: its parameters are not taken."""
    def module(cls, *a, **kw):
        m = cls(*a, **kw)
        calls = []
        m._compiled_call_impl = lambda *x, **k: (calls.append(1), m._call_impl(*x, **k))[1]  # as Module.compile sets it
        return m, calls

    cfg = dict(mi.GPT_CONFIG_124M)
    cfg.update({"emb_dim": 64, "n_layers": 1, "n_heads": 2, "vocab_size": 50, "context_length": 64,
                "drop_rate": 0.0, "impl_type": "manual"})
    model, calls = module(mi.GPTModel, cfg)
    with torch.no_grad():
        mi._last_logits(model.eval(), torch.randint(0, 50, (1, 40)))
    assert calls and not mi._plain(model, mi.GPTModel)
    linear, _ = module(torch.nn.Linear, 4, 4)
    assert not mi._plain(linear, torch.nn.Linear) and mi._plain(torch.nn.Linear(4, 4), torch.nn.Linear)
