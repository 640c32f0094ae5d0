"""The row kernels around the GEMMs of a forward (csrc/elementwise.hip,
csrc/rope.hip): RMSNorm on vector pieces against float64 at the edges of what
stays in registers, SwiGLU on ragged strides, and forwards whose products are
split over K (their partials added by the consuming kernel) against the
module path, whose products choose their own splits, at every row count where
the tile or the split changes.
"""

import dataclasses

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
PAST = 40  # rows cached before the forward under test


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,hidden", [(1, 4), (3, 8), (2, 12), (5, 896), (1, 1000), (7, 3584), (2, 4096),
                                         (2, 8192), (3, 8200), (2, 8196), (1, 20000)])
def test_rmsnorm_matches_float64(rows, hidden, dtype):
    """Rows of 1 to 20,000 elements: whole pieces kept in registers (up to
    8,192 bf16 / 4,096 fp32 elements), read twice past that, and element by
    element when they are not whole 16-byte pieces. Bar: the fp32 sum of
    squares is off by at most hidden 2^-24 relative, half of it after the
    root, a few more roundings, and the output's own rounding."""
    from minitp import kernels as K

    g = torch.Generator(device=DEV).manual_seed(hidden)
    x = (torch.randn(rows, hidden, generator=g, device=DEV) * 3).to(dtype)
    w = (1 + 0.1 * torch.randn(hidden, generator=g, device=DEV)).to(dtype)
    xd = x.double()
    ref = xd * torch.rsqrt(xd.pow(2).mean(-1, keepdim=True) + 1e-6) * w.double()
    got = K.rmsnorm(x, w, 1e-6).double()
    eps = 2.0 ** -24 * (hidden / 2 + 8) + (2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -24)
    assert ((got - ref).abs() <= 2 * eps * ref.abs() + 1e-30).all()


@pytest.mark.parametrize("hidden", [896, 2048, 3584, 8192])
def test_rmsnorm_f32_sums_add_little_error(hidden):
    """The relative 2-norm of the error against what the same fp32 steps give
    with an exact sum of squares (its rounding alone): a fp32 sum's last
    levels may add 6 % to it (four sums in pairs: 4 %; a chain of eight: 9 %)."""
    from minitp import kernels as K

    got_err = ref_err = 0.0
    for seed in range(6):
        g = torch.Generator(device=DEV).manual_seed(seed)
        x = torch.randn(2000, hidden, generator=g, device=DEV)
        w = torch.randn(hidden, generator=g, device=DEV)
        xd = x.double()
        want = xd * torch.rsqrt(xd.pow(2).mean(-1, keepdim=True) + 1e-6) * w.double()
        total = (x * x).double().sum(-1, keepdim=True).float()
        steps = (x * (1.0 / torch.sqrt(total / hidden + 1e-6))) * w
        got_err += (K.rmsnorm(x, w, 1e-6).double() - want).pow(2).sum().item()
        ref_err += (steps.double() - want).pow(2).sum().item()
    assert got_err <= 1.06 ** 2 * ref_err, (got_err / ref_err) ** 0.5


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,n,pad", [(1, 8, 0), (3, 24, 8), (5, 130, 2), (257, 4864, 0), (2, 12, 4)])
def test_silu_mul_matches_float64(rows, n, pad, dtype):
    from minitp import kernels as K

    g = torch.Generator(device=DEV).manual_seed(n)
    wide = torch.randn(rows, 2 * n + pad, generator=g, device=DEV).to(dtype) * 4
    gate, up = wide[:, :n], wide[:, n:2 * n]
    ref = torch.nn.functional.silu(gate.double()) * up.double()
    got = K.silu_mul(gate, up).double()
    eps = 2 * 2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -21
    assert ((got - ref).abs() <= 2 * eps * ref.abs() + 1e-30).all()


@pytest.mark.parametrize("dtype,atol", [(torch.float32, 2e-5), (torch.bfloat16, 0.05)])
@pytest.mark.parametrize("batch,tokens", [(2, 1), (3, 1), (31, 1), (33, 1), (48, 1), (65, 1), (1, 31), (2, 17),
                                          (1, 70), (3, 100), (2, 400), (1, 3), (2, 2), (1, 4)])
@pytest.mark.parametrize("shape", ["05b", "7b"])
def test_forward_matches_the_module_path(shape, batch, tokens, dtype, atol):
    """Two layers at the model's widths on a cache already holding PAST rows.
    The bars are those of the model tests (module path against native)."""
    from minitp import synthetic
    from minitp.generation import make_kv_cache

    full = synthetic.QWEN05B if shape == "05b" else synthetic.QWEN7B
    cfg = dataclasses.replace(full, num_hidden_layers=2, vocab_size=2048, max_position_embeddings=512)
    model = synthetic.build_synthetic_model(cfg, dtype=dtype, device=DEV, seed=0)
    ids = synthetic.synthetic_prompt(cfg.vocab_size, batch, PAST + tokens, seed=1, device=DEV)
    out = []
    for rotary in (True, False):  # False: the module path
        model.use_rotary_cache = rotary
        kv = make_kv_cache(model, batch, PAST + tokens, init="zeros")
        model(ids[:, :PAST], kv_cache=kv)
        pos = torch.arange(PAST, PAST + tokens, device=DEV)
        logits = model(ids[:, PAST:], positions=pos, kv_cache=kv)
        out.append((logits.float(), kv.k[1].float(), kv.v[1].float()))
    for a, b in zip(*out):
        torch.testing.assert_close(a, b, atol=atol, rtol=0.02 if dtype == torch.bfloat16 else 2e-5)


@pytest.mark.parametrize("dtype,atol", [(torch.float32, 2e-5), (torch.bfloat16, 0.05)])
@pytest.mark.parametrize("batch,tokens", [(40, 1), (1, 33), (1, 300)])
def test_forward_takes_a_final_norm_of_any_alignment(batch, tokens, dtype, atol):
    """A final RMSNorm weight that starts one element past a 16-byte boundary
    (the last down projection's partials cannot be added by the vector
    kernel then): the module path's logits."""
    from minitp import synthetic
    from minitp.generation import make_kv_cache

    cfg = dataclasses.replace(synthetic.QWEN05B, num_hidden_layers=2, vocab_size=2048, max_position_embeddings=512)
    model = synthetic.build_synthetic_model(cfg, dtype=dtype, device=DEV, seed=0)
    weight = model.model.norm.weight
    store = torch.empty(weight.numel() + 1, dtype=dtype, device=DEV)
    store[1:] = 1 + 0.1 * torch.randn(weight.numel(), generator=torch.Generator(device=DEV).manual_seed(2), device=DEV)
    model.model.norm.weight = torch.nn.Parameter(store[1:], requires_grad=False)
    ids = synthetic.synthetic_prompt(cfg.vocab_size, batch, PAST + tokens, seed=1, device=DEV)
    out = []
    for rotary in (True, False):  # False: the module path
        model.use_rotary_cache = rotary
        kv = make_kv_cache(model, batch, PAST + tokens, init="zeros")
        model(ids[:, :PAST], kv_cache=kv)
        out.append(model(ids[:, PAST:], positions=torch.arange(PAST, PAST + tokens, device=DEV), kv_cache=kv).float())
    torch.testing.assert_close(*out, atol=atol, rtol=0.02 if dtype == torch.bfloat16 else 2e-5)
