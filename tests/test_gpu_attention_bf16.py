"""bf16 prompt attention at the edges of its forms (csrc/attention.hip): 64- and
128-query blocks, one or two groups of waves over the key tiles (a group
without a visible key, an odd tile left over), query and key counts around
16, 64 and 128, rows past the last key poisoned.

Bar: the output's own rounding (2^-9 of values up to 4) and P rounded to bf16
(2^-9 of the attention-weighted |V|, at most 4): twice their sum, 3e-2.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("d,hq,hkv", [(32, 4, 2), (64, 14, 2), (128, 28, 4), (16, 4, 2)])
@pytest.mark.parametrize("rows", [0, 1100])  # cache capacity: the keys and a few rows, or more
@pytest.mark.parametrize("t,cache_len", [(2, 0), (17, 47), (64, 0), (65, 63), (128, 1), (130, 64), (200, 700),
                                         (1000, 0), (500, 129), (447, 0), (448, 0), (2, 446), (70, 378)])
def test_prefill_attention_bf16_matches_float64(t, cache_len, rows, d, hq, hkv):
    from minitp import kernels as K

    n = cache_len + t
    g = torch.Generator(device=DEV).manual_seed(t * 31 + cache_len + d)
    q = torch.randn(1, t, hq, d, generator=g, device=DEV).bfloat16()
    kc = torch.full((1, hkv, max(n + 5, rows), d), float("nan"), device=DEV, dtype=torch.bfloat16)
    vc = torch.full_like(kc, float("nan"))
    kc[:, :, :n] = torch.randn(1, hkv, n, d, generator=g, device=DEV).bfloat16()
    vc[:, :, :n] = torch.randn(1, hkv, n, d, generator=g, device=DEV).bfloat16()
    out = K.attention(q, kc, vc, cache_len).view(1, t, hq, d).double()
    kk = kc[:, :, :n].double().repeat_interleave(hq // hkv, 1)
    vv = vc[:, :, :n].double().repeat_interleave(hq // hkv, 1)
    s = (q.double().transpose(1, 2) @ kk.transpose(-1, -2).contiguous()) / d ** 0.5
    mask = torch.arange(n, device=DEV)[None, :] > cache_len + torch.arange(t, device=DEV)[:, None]
    ref = (s.masked_fill(mask, float("-inf")).softmax(-1) @ vv).transpose(1, 2)
    assert torch.isfinite(out).all()
    assert (out - ref).abs().max().item() <= 3e-2


@pytest.mark.parametrize("ctx", [1, 33, 511, 1100, 2600])
@pytest.mark.parametrize("b,hq,hkv,d", [(12, 28, 4, 128), (100, 14, 2, 64), (129, 4, 2, 128), (17, 16, 2, 64)])
def test_batched_decode_attention_bf16_split_counts(ctx, b, hq, hkv, d):
    """The grouped decode form at unit counts that do not divide the CUs (one
    to five splits, the last one shorter or empty), groups of 2, 7 and 8. The
    bar adds the output's rounding and P's, each 2^-8 of what it rounds."""
    from minitp import kernels as K

    g = torch.Generator(device=DEV).manual_seed(ctx + b)
    q = torch.randn(b, 1, hq, d, generator=g, device=DEV).bfloat16()
    kc = torch.full((b, hkv, ctx + 3, d), float("nan"), device=DEV, dtype=torch.bfloat16)
    vc = torch.full_like(kc, float("nan"))
    kc[:, :, :ctx] = torch.randn(b, hkv, ctx, d, generator=g, device=DEV).bfloat16()
    vc[:, :, :ctx] = torch.randn(b, hkv, ctx, d, generator=g, device=DEV).bfloat16()
    out = K.attention(q, kc, vc, ctx - 1).view(b, 1, hq, d).double().transpose(1, 2)
    kk, vv = (x[:, :, :ctx].double().repeat_interleave(hq // hkv, 1) for x in (kc, vc))
    p = ((q.double().transpose(1, 2) @ kk.transpose(-1, -2).contiguous()) / d ** 0.5).softmax(-1)
    ref, ref_abs = p @ vv, p @ vv.abs()
    assert torch.isfinite(out).all()
    assert ((out - ref).abs() <= (ref.abs() + ref_abs) * 2 ** -8 + 1e-6).all()
