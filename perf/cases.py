"""Performance cases of the Qwen2 token loop, through its public entry points.

Each case is one call that a program using this framework makes: a decode step
or a prompt prefill of ``GenerationState`` on the native whole-model path, or
the forward of one module (attention, MLP, LM head, RMSNorm) that a program
composes itself. Shapes are the two model shapes of ``minitp.synthetic``
(whole, or with fewer layers where one layer stands for all of them), sizes
run from a single row to the 4 x 4096 prompt, in bf16 and in fp32 (the type
the greedy ids are pinned in).

Weights are N(0, 0.02), biases N(0, 0.02), RMSNorm weights around 1, hidden
states N(0, 1) as a norm leaves them, prompt ids uniform over the vocabulary,
and a cache that is filled before the call holds rows of the spread that the
QKV projection gives.
"""

from __future__ import annotations

import dataclasses
import math
import os
import random
import sys

import torch

_PKG = os.path.join(os.getcwd(), "mini-tp_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

# hidden, intermediate, layers, query heads, KV heads, head dim, vocabulary,
# tied head: the shapes of minitp.synthetic.SHAPES, spelled out because
# exact() and work() use none of the package's code
DIMS = {
    "qwen2.5-0.5b": (896, 4864, 24, 14, 2, 64, 151936, True),
    "qwen2.5-7b": (3584, 18944, 28, 28, 4, 128, 152064, False),
}
EPS, THETA = 1e-6, 1e6
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
DEV = "cuda"


def listed() -> list[dict]:
    return [
        # one RMSNorm of a decode row, called by itself: the smallest call
        _case("norm-row", "norm", "qwen2.5-0.5b", "bf16", batch=1, tokens=1),
        # one token of a chat with the small model, 256 positions cached (its
        # 128 + 256 workload half way)
        _case("decode-0.5b", "decode", "qwen2.5-0.5b", "bf16", layers=24, batch=1, cached=256),
        # one token for 32 sequences at once, 2,300 positions cached each
        # (the 2048 + 512 workload half way)
        _case("decode-0.5b-b32", "decode", "qwen2.5-0.5b", "bf16", layers=24, batch=32, cached=2300),
        # one token of the large model (its 512 + 256 workload), a quarter of
        # its layers and the untied head
        _case("decode-7b", "decode", "qwen2.5-7b", "bf16", layers=7, batch=1, cached=640),
        # one token for an odd handful of sequences in fp32
        _case("decode-0.5b-fp32-b3", "decode", "qwen2.5-0.5b", "fp32", layers=24, batch=3, cached=777),
        # time to first token of the small model's 128-token prompt
        _case("prefill-0.5b-128", "prefill", "qwen2.5-0.5b", "bf16", layers=24, batch=1, tokens=128),
        # a ragged middle-sized prompt on the large model's layers
        _case("prefill-7b-433", "prefill", "qwen2.5-7b", "bf16", layers=4, batch=1, tokens=433),
        # the long-prompt workload, 4 x 4096 tokens, on two layers: the largest
        _case("prefill-7b-4x4096", "prefill", "qwen2.5-7b", "bf16", layers=2, batch=4, tokens=4096),
        # three ragged prompts in fp32
        _case("prefill-0.5b-fp32-3x333", "prefill", "qwen2.5-0.5b", "fp32", layers=6, batch=3, tokens=333),
        # one chunk of a long document: 512 new tokens after 1,500 cached ones
        _case("attention-7b-chunk", "attention", "qwen2.5-7b", "bf16", batch=1, tokens=512, cached=1500),
        # the MLP of a batch of short prompts, an odd number of rows
        _case("mlp-0.5b-7x157", "mlp", "qwen2.5-0.5b", "bf16", batch=7, tokens=157),
        # logits of every position of a short text (scoring)
        _case("head-0.5b-2x97", "head", "qwen2.5-0.5b", "bf16", batch=2, tokens=97),
    ]


def _case(name: str, kind: str, shape: str, dtype: str, *, layers: int = 1, batch: int, tokens: int = 1,
          cached: int = 0) -> dict:
    return {"name": name, "kind": kind, "shape": shape, "dtype": dtype, "layers": layers, "batch": batch,
            "tokens": tokens, "cached": cached}


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng: random.Random) -> dict:
    """One more case of the same ranges: every kind, shape and type, batches of
    1 to 48 sequences, 1 to 4096 positions, no dearer than the largest listed."""
    limit = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["decode", "decode", "prefill", "prefill", "attention", "mlp", "head", "norm"])
        shape = rng.choice(sorted(DIMS))
        case = {"kind": kind, "shape": shape, "dtype": rng.choice(["bf16", "bf16", "bf16", "fp32"]), "layers": 1,
                "batch": _log_int(rng, 1, 48), "tokens": 1, "cached": 0}
        if kind == "decode":
            case["layers"] = rng.randint(1, 24 if shape == "qwen2.5-0.5b" else 7)
            case["cached"] = _log_int(rng, 1, 4096)
        elif kind == "prefill":
            case["layers"] = rng.randint(1, 4)
            case["batch"] = _log_int(rng, 1, 8)
            case["tokens"] = _log_int(rng, 2, 4096)
        elif kind == "attention":
            case["batch"] = _log_int(rng, 1, 8)
            case["tokens"] = _log_int(rng, 1, 2048)
            case["cached"] = rng.choice([0, _log_int(rng, 1, 2048)])
        else:
            case["tokens"] = _log_int(rng, 1, 512 if kind == "head" else 2048)
            if kind == "head":
                case["batch"] = _log_int(rng, 1, 4)
        if _cost(case) <= limit:
            return case


def _cost(case: dict) -> float:
    """Seconds at 1 PFLOP/s bf16 (a sixteenth of that in fp32) plus 4 TB/s."""
    w = work(case)
    return w["flops"] / (1e15 if case["dtype"] == "bf16" else 6e13) + w["bytes"] / 4e12


# ---------------------------------------------------------------------------
# inputs (made with torch alone, so that exact() sees the same ones)


def _gen(seed: int, stream: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed * 1009 + stream)


def _normal(g: torch.Generator, shape, dtype: torch.dtype, std: float, mean: float = 0.0) -> torch.Tensor:
    return torch.empty(shape, dtype=torch.float32, device=DEV).normal_(mean, std, generator=g).to(dtype)


def _weights(case: dict, seed: int) -> dict[str, torch.Tensor]:
    """The case's parameters under the model's state-dict names."""
    h, inter, _, hq, hkv, d, vocab, tied = DIMS[case["shape"]]
    dt, kind, g = DTYPES[case["dtype"]], case["kind"], _gen(seed, 1)
    whole = kind in ("decode", "prefill")
    sd: dict[str, torch.Tensor] = {}
    if whole:
        sd["model.embed_tokens.weight"] = _normal(g, (vocab, h), dt, 0.02)
        sd["lm_head.weight"] = sd["model.embed_tokens.weight"] if tied else _normal(g, (vocab, h), dt, 0.02)
    elif kind == "head":
        sd["weight"] = _normal(g, (vocab, h), dt, 0.02)
    if whole or kind == "norm":
        sd["model.norm.weight" if whole else "weight"] = _normal(g, (h,), dt, 0.1, 1.0)
    for i in range(case["layers"]):
        p = f"model.layers.{i}." if whole else ""
        if whole:
            sd[p + "input_layernorm.weight"] = _normal(g, (h,), dt, 0.1, 1.0)
            sd[p + "post_attention_layernorm.weight"] = _normal(g, (h,), dt, 0.1, 1.0)
        a, m = (p + "self_attn.", p + "mlp.") if whole else ("", "")
        if whole or kind == "attention":
            sd[a + "qkv_proj.weight"] = _normal(g, ((hq + 2 * hkv) * d, h), dt, 0.02)
            sd[a + "qkv_proj.bias"] = _normal(g, ((hq + 2 * hkv) * d,), dt, 0.02)
            sd[a + "o_proj.weight"] = _normal(g, (h, hq * d), dt, 0.02)
        if whole or kind == "mlp":
            sd[m + "gate_up_proj.weight"] = _normal(g, (2 * inter, h), dt, 0.02)
            sd[m + "down_proj.weight"] = _normal(g, (h, inter), dt, 0.02)
    return sd


def _ids(case: dict, seed: int) -> torch.Tensor:
    return torch.randint(0, DIMS[case["shape"]][6], (case["batch"], case["cached"] + case["tokens"]),
                         generator=_gen(seed, 2), device=DEV)


def _hidden(case: dict, seed: int) -> torch.Tensor:
    h = DIMS[case["shape"]][0]
    return _normal(_gen(seed, 3), (case["batch"], case["tokens"], h), DTYPES[case["dtype"]], 1.0)


def _cached_rows(case: dict, seed: int, layer: int) -> tuple[torch.Tensor, torch.Tensor]:
    """K and V rows [B, Hkv, cached, D] that earlier calls left in the cache."""
    h, _, _, _, hkv, d, _, _ = DIMS[case["shape"]]
    shape, g = (case["batch"], hkv, case["cached"], d), _gen(seed, 16 + layer)
    std, dt = 0.02 * math.sqrt(h), DTYPES[case["dtype"]]
    return _normal(g, shape, dt, std), _normal(g, shape, dt, std)


# ---------------------------------------------------------------------------
# the program's side


def prepare(case: dict, seed: int) -> dict:
    from minitp.distributed.context import ParallelContext
    from minitp.kv_cache import KVCache
    from minitp.rope import RotaryEmbedding
    from minitp.synthetic import SHAPES

    kind, b, t, cached = case["kind"], case["batch"], case["tokens"], case["cached"]
    dt = DTYPES[case["dtype"]]
    cfg = dataclasses.replace(SHAPES[case["shape"]], num_hidden_layers=case["layers"])
    ctx = ParallelContext(0, 0, 1, 0, 1, torch.device(DEV), None)
    module = _module(kind, cfg, ctx)
    module.load_state_dict(_weights(case, seed), assign=True)
    module = module.eval().requires_grad_(False)
    state = {"case": case, "module": module}
    if kind in ("decode", "prefill", "attention"):
        # a cache slot that the program keeps for the sequences it serves
        kv = KVCache(case["layers"], b, cfg.num_key_value_heads, cfg.head_dim, cached + t + 1, dt, torch.device(DEV),
                     init="zeros")
        for i in range(case["layers"]):
            if cached:
                k, v = _cached_rows(case, seed, i)
                kv.k[i][:, :, :cached] = k
                kv.v[i][:, :, :cached] = v
        state["kv"] = kv
    if kind == "decode":
        from minitp.generation import GenerationState

        if cfg.tie_word_embeddings:
            module.lm_head.weight = module.model.embed_tokens.weight
        ids = _ids(case, seed)
        state["gen"] = GenerationState(module, ids, 1, kv=kv)
        module.program()
    elif kind == "prefill":
        if cfg.tie_word_embeddings:
            module.lm_head.weight = module.model.embed_tokens.weight
        state["ids"] = _ids(case, seed)
        module.program()
    else:
        state["x"] = _hidden(case, seed)
    if kind == "attention":
        state["rotary"] = RotaryEmbedding(cfg.head_dim, cfg.rope_theta, cached + t, torch.device(DEV))
        state["positions"] = torch.arange(cached, cached + t, device=DEV)
    return state


def _module(kind: str, cfg, ctx):
    from minitp.attention import TPQwen2Attention
    from minitp.layer import RMSNorm, TPQwen2ForCausalLM
    from minitp.mlp import TPQwen2MLP
    from minitp.parallel.embedding import VocabParallelLMHead

    with torch.device("meta"):
        if kind in ("decode", "prefill"):
            return TPQwen2ForCausalLM(cfg, ctx, init_weights=False)
        if kind == "attention":
            return TPQwen2Attention(cfg, ctx, init_weights=False)
        if kind == "mlp":
            return TPQwen2MLP(cfg, ctx, init_weights=False)
        if kind == "head":
            return VocabParallelLMHead(cfg.hidden_size, cfg.vocab_size, ctx, init_weights=False)
        return RMSNorm(cfg.hidden_size, cfg.rms_norm_eps, init_weights=False)


@torch.inference_mode()
def run(state: dict):
    case, module = state["case"], state["module"]
    kind, cached, t = case["kind"], case["cached"], case["tokens"]
    if kind == "decode":
        # one step of a running generation, from the same cursor each time
        st, kv = state["gen"], state["kv"]
        st.cursor, kv.seq_len = cached, cached
        tok = st.out_ids[:, cached]
        pos = st.append(tok)
        logits = st.decode_step(tok, pos)
        return {"logits": logits, "k": _new_rows(kv.k, cached, 1), "v": _new_rows(kv.v, cached, 1)}
    if kind == "prefill":
        # a new prompt into a free cache slot, up to its first token's logits
        from minitp.generation import GenerationState

        kv = state["kv"]
        kv.seq_len = 0
        st = GenerationState(module, state["ids"], 1, kv=kv, prefill_logits="last")
        logits = st.prefill()
        return {"logits": logits, "k": _new_rows(kv.k, 0, t), "v": _new_rows(kv.v, 0, t)}
    if kind == "attention":
        kv = state["kv"]
        kv.seq_len = cached
        out = module(state["x"], state["positions"], kv, 0, state["rotary"])
        return {"out": out, "k": _new_rows(kv.k, cached, t), "v": _new_rows(kv.v, cached, t)}
    return module(state["x"])


def _new_rows(layers: list[torch.Tensor], start: int, count: int) -> list[torch.Tensor]:
    return [c[:, :, start:start + count] for c in layers]


# ---------------------------------------------------------------------------
# what a pass cannot do without, and what its outputs should be


def work(case: dict) -> dict:
    h, inter, _, hq, hkv, d, vocab, _ = DIMS[case["shape"]]
    es = 2 if case["dtype"] == "bf16" else 4
    kind, b, t, cached, layers = case["kind"], case["batch"], case["tokens"], case["cached"], case["layers"]
    rows = b * t
    qkv_n, q_n = (hq + 2 * hkv) * d, hq * d
    attn_params, mlp_params = qkv_n * h + h * q_n, 3 * inter * h
    keys = t * cached + t * (t + 1) // 2  # (query, key) pairs of one sequence and head
    attn_flops = 2 * rows * attn_params + 4 * b * hq * d * keys
    # cached rows read, new rows written
    cache_bytes = 2 * b * hkv * d * (cached + t) * es
    if kind in ("decode", "prefill"):
        params = layers * (attn_params + qkv_n + mlp_params + 2 * h) + h + vocab * h
        flops = layers * (attn_flops + 2 * rows * mlp_params) + 2 * b * vocab * h
        nbytes = params * es + rows * (h * es + 8) + layers * cache_bytes + b * vocab * es
    elif kind == "attention":
        flops = attn_flops
        nbytes = (attn_params + qkv_n + 2 * rows * h) * es + cache_bytes
    elif kind == "mlp":
        flops, nbytes = 2 * rows * mlp_params, (mlp_params + 2 * rows * h) * es
    elif kind == "head":
        flops, nbytes = 2 * rows * vocab * h, (vocab * h + rows * (h + vocab)) * es
    else:
        flops, nbytes = 4 * rows * h, (h + 2 * rows * h) * es
    return {"bytes": int(nbytes), "flops": int(flops)}


def tolerance(case: dict) -> dict:
    # about four times the distance from exact() that was measured: fp32
    # 2.8e-6 after 24 layers; bf16 modules 0.002-0.0046; bf16 models, whose
    # layers carry on what earlier ones left, 0.007 after one layer, 0.014
    # after two, 0.02 after four to seven, 0.03 after 24
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    if case["kind"] in ("decode", "prefill"):
        return {"rel": 2.5e-2 * math.sqrt(1 + case["layers"])}
    return {"rel": 1.6e-2}


def _linear64(x: torch.Tensor, w: torch.Tensor, bias: torch.Tensor | None = None) -> torch.Tensor:
    """x W^T (+ bias) in 64 bits, the weight widened a block of rows at a time."""
    out = torch.empty(*x.shape[:-1], w.shape[0], dtype=torch.float64, device=x.device)
    for lo in range(0, w.shape[0], 16384):
        out[..., lo:lo + 16384] = x @ w[lo:lo + 16384].double().t()
    return out if bias is None else out + bias.double()


def _norm64(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x: torch.Tensor, positions: torch.Tensor) -> torch.Tensor:
    """Rotation of [B, H, T, D] by the fp32 angle tables that the model defines."""
    d = x.shape[-1]
    inv = 1.0 / (THETA ** (torch.arange(0, d, 2, dtype=torch.float32) / d))
    ang = positions.cpu().float()[:, None] * inv[None, :]
    ang = torch.cat([ang, ang], dim=-1)
    cos, sin = ang.cos().double().to(x.device), ang.sin().double().to(x.device)
    half = torch.cat([-x[..., d // 2:], x[..., :d // 2]], dim=-1)
    return x * cos + half * sin


def _attention64(x, sd, prefix, case, cache):
    _, _, _, hq, hkv, d, _, _ = DIMS[case["shape"]]
    b, t, cached = case["batch"], case["tokens"], case["cached"]
    y = _linear64(x, sd[prefix + "qkv_proj.weight"], sd[prefix + "qkv_proj.bias"]).view(b, t, hq + 2 * hkv, d)
    y = y.transpose(1, 2)
    pos = torch.arange(cached, cached + t)
    q, k = _rope64(y[:, :hq], pos), _rope64(y[:, hq:hq + hkv], pos)
    v = y[:, hq + hkv:]
    ka, va = torch.cat([cache[0].double(), k], 2), torch.cat([cache[1].double(), v], 2)
    out = torch.empty(b, t, hq, d, dtype=torch.float64, device=x.device)
    keys = torch.arange(cached + t, device=x.device)
    for i in range(b):
        for head in range(hq):
            kh, vh = ka[i, head // (hq // hkv)], va[i, head // (hq // hkv)]
            s = (q[i, head] @ kh.t()) / math.sqrt(d)
            s.masked_fill_(keys[None, :] > pos.to(x.device)[:, None], float("-inf"))
            out[i, :, head] = torch.softmax(s, -1) @ vh
    return _linear64(out.reshape(b, t, hq * d), sd[prefix + "o_proj.weight"]), k, v


def _mlp64(x, sd, prefix):
    g, u = _linear64(x, sd[prefix + "gate_up_proj.weight"]).chunk(2, -1)
    return _linear64(torch.nn.functional.silu(g) * u, sd[prefix + "down_proj.weight"])


@torch.inference_mode()
def exact(case: dict, seed: int):
    if work(case)["flops"] > 2.5e13:
        return None
    kind, sd = case["kind"], _weights(case, seed)
    if kind in ("decode", "prefill"):
        ids = _ids(case, seed)[:, case["cached"]:]
        x = sd["model.embed_tokens.weight"][ids].double()
        ks, vs = [], []
        for i in range(case["layers"]):
            p = f"model.layers.{i}."
            a, k, v = _attention64(_norm64(x, sd[p + "input_layernorm.weight"]), sd, p + "self_attn.", case,
                                   _cached_rows(case, seed, i))
            ks.append(k)
            vs.append(v)
            x = x + a
            x = x + _mlp64(_norm64(x, sd[p + "post_attention_layernorm.weight"]), sd, p + "mlp.")
        logits = _linear64(_norm64(x[:, -1:], sd["model.norm.weight"]), sd["lm_head.weight"])
        return {"logits": logits, "k": ks, "v": vs}
    x = _hidden(case, seed).double()
    if kind == "attention":
        out, k, v = _attention64(x, sd, "", case, _cached_rows(case, seed, 0))
        return {"out": out, "k": [k], "v": [v]}
    if kind == "mlp":
        return _mlp64(x, sd, "")
    if kind == "head":
        return _linear64(x, sd["weight"])
    return _norm64(x, sd["weight"])
