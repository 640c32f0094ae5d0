"""The MFMA GEMM of prompts and batched decode (csrc/gemm.hip) at the edges of
its tiles: rows and columns just below, at and past each tile shape, K tails
shorter than a stage and shorter than the ring, and shapes on both sides of
the tile-choice rule (64 x 64 up to 256 x 128).

Bar: against float64 products. fp32 sums of K terms in any order are off by
at most K 2^-24 sum |x_k w_k| (twice that for fp32 operands, whose products
round too), and a bf16 output is off by half a step more (2^-9 relative);
both are doubled here.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"

SHAPES = [
    (33, 64, 8),          # one stage, one chunk of it
    (63, 130, 72),        # ragged columns (not a multiple of 4), K tail of one chunk
    (64, 896, 896),
    (65, 1152, 200),
    (100, 77, 264),       # odd width
    (129, 4608, 1000),
    (194, 9728, 896),
    (257, 640, 4864),     # long K on few tiles
    (433, 3584, 1096),    # 64 x 128 and 128 x 128 tiles at 7B widths
    (700, 9728, 520),
    (2000, 3584, 384),    # 256 x 128 tiles
    (40, 3584, 18944),    # split over K: few tiles, long K
    (100, 896, 4864),
    (17, 130, 4864),      # (fp32: split, ragged columns)
    (3, 896, 904),        # (fp32: the register GEMVs of 2-4 rows, to their last chunk)
    (4, 897, 1024),
    (3, 70, 1032),
    (2, 96, 4104),
    (4, 896, 4864),
    (2, 1153, 5120),
    (3, 64, 5128),
    (3, 18433, 1032),     # (fp32: the GEMM's side of the line at 18,432 rows of the weight)
    (4, 18432, 2560),
    (2, 130, 8200),       # (bf16: two rows past the GEMVs, split over K)
    (1, 70, 20488),
]


def _bound(ref, x, w, dtype, k):
    mag = x.double().abs() @ w.double().abs().t()
    eps = 2.0 ** -24 * k * (2 if dtype == torch.float32 else 1)
    return 2 * (eps * mag + (2.0 ** -9 * ref.abs() if dtype == torch.bfloat16 else 2.0 ** -24 * ref.abs())) + 1e-30


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_linear_matches_float64(m, n, k, dtype):
    """Plain product, with and without bias, from rows inside a wider buffer
    whose other columns are NaN (nothing past K may reach a sum)."""
    from minitp import kernels as K

    g = torch.Generator(device=DEV).manual_seed(m * 7 + n + k)
    wide = torch.full((m, k + 64), float("nan"), dtype=dtype, device=DEV)
    wide[:, :k] = torch.randn(m, k, generator=g, device=DEV).to(dtype)
    x = wide[:, :k]
    w = (torch.randn(n, k, generator=g, device=DEV) * 0.05).to(dtype)
    bias = torch.randn(n, generator=g, device=DEV).to(dtype)
    ref = x.double() @ w.double().t()
    for b, r in ((None, ref), (bias, ref + bias.double())):
        got = K.linear(x, w, b).double()
        assert torch.isfinite(got).all()
        over = ((got - r).abs() - _bound(r, x, w, dtype, k)).max().item()
        assert over <= 0, (b is not None, over)


@pytest.mark.parametrize("m,n,k", [(65, 1152, 200), (433, 3584, 1096), (40, 1792, 9480)])
def test_linear_resid_matches_float64(m, n, k):
    from minitp import _native as N
    from minitp import kernels as K

    g = torch.Generator(device=DEV).manual_seed(m + n)
    x = torch.randn(m, k, generator=g, device=DEV).bfloat16()
    w = (torch.randn(n, k, generator=g, device=DEV) * 0.05).bfloat16()
    aux = torch.randn(m, n, generator=g, device=DEV).bfloat16()
    prod = x.double() @ w.double().t()
    got = K.linear(x, w, epilogue=N.EPI_RESID, aux=aux).double()
    ref = prod + aux.double()
    bar = _bound(prod, x, w, torch.bfloat16, k) + 2 * 2.0 ** -9 * ref.abs()
    over = ((got - ref).abs() - bar).max().item()
    assert over <= 0, over


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,n,k", [(1, 64, 64), (2, 4864, 896), (5, 130, 72), (33, 77, 200), (64, 4864, 896),
                                   (65, 96, 1000), (130, 1001, 520), (300, 4864, 264), (700, 2368, 136)])
def test_gate_up_swiglu_matches_float64(m, n, k, dtype):
    """Bar: the products' bars through silu(g) u (|silu'| < 1.1), plus the
    roundings of g, u, silu(g) and the output."""
    from minitp import _native as N
    from minitp import kernels as K

    g = torch.Generator(device=DEV).manual_seed(m + 3 * n + k)
    x = torch.randn(m, k, generator=g, device=DEV).to(dtype)
    w = (torch.randn(2 * n, k, generator=g, device=DEV) * 0.05).to(dtype)
    y = x.double() @ w.double().t()
    gate, up = y[:, :n], y[:, n:]
    b = _bound(y, x, w, dtype, k)
    ref = torch.nn.functional.silu(gate) * up
    unit = 2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -22
    bar = 1.1 * b[:, :n] * up.abs() + torch.nn.functional.silu(gate).abs() * b[:, n:] + 4 * unit * ref.abs() + 1e-6 * (
        dtype == torch.bfloat16)
    outs = [K.gate_up_swiglu(x, w)]
    if dtype == torch.bfloat16 and m <= 32 and n % 2 == 0:  # the GEMV rows of minitp_linear, any even width
        outs.append(K.linear(x, w, epilogue=N.EPI_SWIGLU))
    for got in outs:
        over = ((got.double() - ref).abs() - 1.01 * bar).max().item()
        assert over <= 0, over


@pytest.mark.parametrize("tokens", [33, 65, 129, 200, 321])
def test_swiglu_forms_agree_with_the_module(tokens):
    """A prompt's gate/up product with SwiGLU in the GEMM's epilogue (the
    native forward) against the module path (product, then SwiGLU), one
    layer at the 0.5B widths: logits and cache rows."""
    import dataclasses

    from minitp import synthetic
    from minitp.generation import make_kv_cache

    cfg = dataclasses.replace(synthetic.QWEN05B, num_hidden_layers=2, vocab_size=4096)
    model = synthetic.build_synthetic_model(cfg, dtype=torch.bfloat16, device=DEV, seed=0)
    ids = synthetic.synthetic_prompt(cfg.vocab_size, 1, tokens, seed=1, device=DEV)
    out = []
    for rotary in (True, False):  # False: the module path
        model.use_rotary_cache = rotary
        kv = make_kv_cache(model, 1, tokens, init="zeros")
        out.append((model(ids, kv_cache=kv).float(), kv.k[1].float()))
    model.use_rotary_cache = True
    for a, b in zip(*out):
        torch.testing.assert_close(a, b, atol=0.05, rtol=0.02)


@pytest.mark.parametrize("m,n,k", [(250, 65700, 200), (194, 65665, 264), (255, 98432, 896), (256, 65664, 1000),
                                   (201, 131001, 8), (195, 80001, 72), (133, 131002, 136)])
def test_linear_of_many_tiles_matches_float64(m, n, k):
    """Products whose blocks walk several tiles on one running ring of stages:
    one row tile, full and not, a last column tile not full, columns not in
    fours, one to sixteen stages a tile (fewer than the ring's and odd counts
    among them), a last round that some blocks sit out; the bar of the plain
    products."""
    test_linear_matches_float64(m, n, k, torch.bfloat16)


@pytest.mark.parametrize("m,n,k", [(433, 64, 64), (33, 40000, 72), (1500, 2001, 128), (64, 2000, 136), (300, 901, 1024),
                                   (64, 37893, 1096), (130, 9731, 896), (64, 50001, 1000), (250, 9730, 1000)])
def test_linear_of_few_stages_matches_float64(m, n, k):
    """Products of at most 16 stages on every tile shape (whole in the ring,
    two to four stages, 64 x 64 to 128 x 128), and one row tile of many
    blocks past that: ragged rows, columns and stages."""
    test_linear_matches_float64(m, n, k, torch.bfloat16)


@pytest.mark.parametrize("m,n,k", [(70, 1001, 104), (129, 9731, 136), (300, 901, 896), (200, 9730, 1000)])
def test_linear_resid_of_few_stages_matches_float64(m, n, k):
    test_linear_resid_matches_float64(m, n, k)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("hidden,inter,heads,kv_heads,head_dim", [(896, 4864, 14, 2, 64), (3584, 18944, 28, 4, 128),
                                                                  (264, 136, 4, 2, 32)])
def test_unfused_projections_give_the_packed_ones_bits(hidden, inter, heads, kv_heads, head_dim, dtype):
    """Row blocks of the packed QKV and gate/up weights as products of their
    own against the packed products, and the MLP with and without its fused
    gate/up: bitwise, at row counts on every form the packed product takes."""
    from minitp.config import ModelConfig
    from minitp.distributed.context import ParallelContext
    from minitp.mlp import TPQwen2MLP
    from minitp.parallel.fused import FusedQKVColumnParallelLinear

    cfg = ModelConfig(hidden, inter, 1, heads, kv_heads, head_dim, 128, 1e-6, 1e6, 64)
    ctx = ParallelContext(0, 0, 1, 0, 1, torch.device(DEV), None)
    g = torch.Generator(device=DEV).manual_seed(hidden)
    with torch.device(DEV):
        qkv = FusedQKVColumnParallelLinear(hidden, heads * head_dim, kv_heads * head_dim, ctx).to(dtype)
        mlp = TPQwen2MLP(cfg, ctx).to(dtype)
    with torch.no_grad():
        for p in [*qkv.parameters(), *mlp.parameters()]:
            p.copy_(torch.randn(p.shape, generator=g, device=DEV) * 0.02)
        for m in (1, 2, 3, 4, 5, 32, 33, 48, 65, 100, 157, 300, 433, 512, 700, 1099, 2100, 4096):
            if dtype == torch.float32 and m * hidden * inter > 1.2e11:
                continue
            x = torch.randn(m, hidden, generator=g, device=DEV).to(dtype)
            assert torch.equal(qkv.project(x), qkv.project(x, fused=False)), ("qkv", m)
            gu = mlp.gate_up_proj
            assert torch.equal(gu.project(x), gu.project(x, fused=False)), ("gate_up", m)
            outs = []
            for mlp.use_fused_gateup in (True, False):
                outs.append(mlp(x))
            assert torch.equal(*outs), ("mlp", m)


@pytest.mark.parametrize("room", [0, 16, 4 << 10])
def test_linear_ws_with_less_than_the_split_workspace(room):
    """A shape that splits over K, its workspace absent or too small: the
    unsplit product."""
    from minitp import _native as N

    m, n, k = 40, 896, 4864
    lib, dt = N.lib(), N.dtype_code(torch.bfloat16)
    need = lib.minitp_linear_workspace_bytes(dt, m, n, k, N.EPI_NONE)
    assert need > room
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn(m, k, generator=g, device=DEV).bfloat16()
    w = (torch.randn(n, k, generator=g, device=DEV) * 0.05).bfloat16()
    ws = torch.empty(max(room, 16), dtype=torch.uint8, device=DEV)
    y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    N.check(lib.minitp_linear_ws(N.stream(), dt, x.data_ptr(), k, w.data_ptr(), None, y.data_ptr(), n, m, n, k,
                                 N.EPI_NONE, None, ws.data_ptr() if room else None, room), "linear")
    ref = x.double() @ w.double().t()
    assert ((y.double() - ref).abs() <= _bound(ref, x, w, torch.bfloat16, k)).all()


@pytest.mark.parametrize("m,n,k,lo", [(40, 130, 264, 1), (300, 896, 520, 3), (33, 64, 4864, 2), (600, 1001, 200, 5)])
def test_linear_into_columns_of_any_alignment(m, n, k, lo):
    """``out`` a column slice whose base is not aligned to the four-column
    stores: the product in the slice, its neighbours untouched."""
    from minitp import kernels as K

    g = torch.Generator(device=DEV).manual_seed(m + n)
    x = torch.randn(m, k, generator=g, device=DEV).bfloat16()
    w = (torch.randn(n, k, generator=g, device=DEV) * 0.05).bfloat16()
    wide = torch.full((m, n + 12), float("nan"), dtype=torch.bfloat16, device=DEV)
    K.linear(x, w, out=wide[:, lo:lo + n])
    ref = x.double() @ w.double().t()
    assert ((wide[:, lo:lo + n].double() - ref).abs() <= _bound(ref, x, w, torch.bfloat16, k)).all()
    assert wide[:, :lo].isnan().all() and wide[:, lo + n:].isnan().all()
