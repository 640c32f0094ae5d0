"""fp32 prompt attention on the matrix cores (csrc/attention.hip) at the edges
of its 16-query strips, 64-query blocks and 32- / 64-key tiles, for every head
dim it serves, with the cache rows past the last key poisoned.

Bar: rounding errors taken as independent, a score of D products carries
about 2^-24 sqrt(D) (7e-7 at D = 128), so each probability that relative
error plus two roundings of the exponential, and an output of values of order
1 the same; five standard deviations over the outputs, twice: 1e-5.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("d", [16, 32, 64, 128])
@pytest.mark.parametrize("t,cache_len", [(2, 0), (15, 1), (16, 16), (17, 31), (33, 33), (63, 64), (64, 0), (65, 127),
                                         (130, 5), (333, 0), (200, 700)])
def test_prefill_attention_f32_matches_float64(t, cache_len, d):
    from minitp import kernels as K

    b, hq, hkv = 2, 6, 2
    g = torch.Generator(device=DEV).manual_seed(t * 31 + cache_len + d)
    q = torch.randn(b, t, hq, d, generator=g, device=DEV)
    n = cache_len + t
    kc = torch.full((b, hkv, n + 5, d), float("nan"), device=DEV)
    vc = torch.full_like(kc, float("nan"))
    kc[:, :, :n] = torch.randn(b, hkv, n, d, generator=g, device=DEV)
    vc[:, :, :n] = torch.randn(b, hkv, n, d, generator=g, device=DEV)
    out = K.attention(q, kc, vc, cache_len).view(b, t, hq, d).double()
    kk = kc[:, :, :n].double().repeat_interleave(hq // hkv, 1)
    vv = vc[:, :, :n].double().repeat_interleave(hq // hkv, 1)
    s = (q.double().transpose(1, 2) @ kk.transpose(-1, -2).contiguous()) / d ** 0.5
    mask = torch.arange(n, device=DEV)[None, :] > cache_len + torch.arange(t, device=DEV)[:, None]
    ref = (s.masked_fill(mask, float("-inf")).softmax(-1) @ vv).transpose(1, 2)
    assert torch.isfinite(out).all()
    assert (out - ref).abs().max().item() <= 1e-5


@pytest.mark.parametrize("t,hq,d", [(64, 28, 128), (40, 14, 64)])
def test_prefill_attention_f32_scores_in_short_chains(t, hq, d):
    """The relative 2-norm of the error. A chain of m sums of products of
    N(0, 1) factors has partial sums of sqrt(k), each rounded by u sqrt(k / 3) (u =
    2^-24): a variance of u^2 m^2 / 6. Four chains of D / 4 and the two levels
    of their sum: u^2 (D^2 / 24 + 2 D / 3), and over the D of the scale that is the
    relative error of a weight, so of an output (the sums over a few dozen keys add
    little): u sqrt(D / 24 + 2 / 3). One chain of D: u sqrt(D / 6), past the bar."""
    from minitp import kernels as K

    errs = []
    for seed in range(4):
        g = torch.Generator(device=DEV).manual_seed(seed)
        q = torch.randn(2, t, hq, d, generator=g, device=DEV)
        kc, vc = (torch.randn(2, 2, t, d, generator=g, device=DEV) for _ in range(2))
        out = K.attention(q, kc, vc, 0).view(2, t, hq, d).double()
        kk, vv = (x.double().repeat_interleave(hq // 2, 1) for x in (kc, vc))
        s = (q.double().transpose(1, 2) @ kk.transpose(-1, -2).contiguous()) / d ** 0.5
        mask = torch.triu(torch.ones(t, t, device=DEV, dtype=torch.bool), 1)
        ref = (s.masked_fill(mask, float("-inf")).softmax(-1) @ vv).transpose(1, 2)
        errs.append(((out - ref).norm() / ref.norm()).item())
    assert sum(errs) / len(errs) <= 1.15 * 2.0 ** -24 * (d / 24 + 2 / 3) ** 0.5, errs


def test_prefill_attention_f32_large_scores():
    """Scores far past the exponential's range, one key per query dominating."""
    from minitp import kernels as K

    t, d = 40, 64
    g = torch.Generator(device=DEV).manual_seed(5)
    q = torch.randn(1, t, 1, d, generator=g, device=DEV) * 40
    k = torch.randn(1, 1, t, d, generator=g, device=DEV) * 40
    v = torch.randn(1, 1, t, d, generator=g, device=DEV)
    out = K.attention(q, k, v, 0).view(t, d)
    s = (q[0, :, 0].double() @ k[0, 0].double().t().contiguous()) / d ** 0.5
    s = s.masked_fill(torch.triu(torch.ones(t, t, device=DEV, dtype=torch.bool), 1), float("-inf"))
    ref = s.softmax(-1) @ v[0, 0].double()
    # scores of order 13,000 carry an absolute error of up to 13,000 x 2^-24 x 8
    assert torch.isfinite(out).all()
    assert (out.double() - ref).abs().max().item() <= 0.05


@pytest.mark.parametrize("dtype,d,t", [(torch.float32, 128, 2), (torch.bfloat16, 128, 3), (torch.bfloat16, 128, 70)])
def test_prefill_attention_past_4_gib_of_keys(dtype, d, t):
    """A head whose rows span more than 4 GiB: zeros but for one key past that
    line (and its image modulo 2^32 bytes), which every query picks."""
    from minitp import kernels as K

    rows = (1 << 32) // (d * dtype.itemsize)
    n = rows + 200 + t
    kc = torch.zeros(1, 1, n, d, dtype=dtype, device=DEV)
    vc = torch.zeros_like(kc)
    q = torch.ones(1, t, 1, d, dtype=dtype, device=DEV)
    at = rows + 100
    kc[0, 0, at] = 64.0  # score 64 sqrt(128): e^-724 is left for the zero keys
    vc[0, 0, at] = torch.arange(d, device=DEV).to(dtype)
    vc[0, 0, at % rows] = -5.0
    out = K.attention(q, kc, vc, n - t).view(t, d)
    assert torch.equal(out, vc[0, 0, at].expand(t, d))
