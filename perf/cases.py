"""The work whose speed is measured: AnchorAttention as its users call it, on one GPU.

Six kinds of work, each through the public entry points that a program calls:

operator  ``anchor_attn(q, k, v, ...)`` on one layer's tensors: what the reference's callers and benchmarks run.
prefill   the attention plug on a prompt of any length, as a patched model's layers call it: whole big blocks go
          through the operator, the ragged tail (or all of a prompt shorter than a big block) through dense attention.
decode    the plug with one new token per sequence against a key/value cache (a batch's prompts differ in length: left-padded).
padded    the plug on a left-padded batch with its boolean mask.
dense     ``dense_causal_attention``, the dense baseline (pattern "dense").
model     the forward of a patched Hugging Face Llama of two layers with random weights: logits and cache.

Head counts and sizes are those of the repository's configurations, tests and benchmark (Llama-3.1-8B, Qwen2.5-7B,
Llama-3.2-1B and Qwen2.5-0.5B layer shapes).  Inputs are the synthetic long-context tensors of the benchmark, drawn on
the GPU: RoPE'd normal queries and keys with an attention sink and stripe keys ("shared": a component that all queries of
a KV group share makes these score far above the rest, so few keys are selected; "literal": no shared component, nearly
every key is selected).
"""
import math
import os
import sys
import types

import torch

sys.path.insert(0, os.path.abspath("anchor-attention_amd"))

from anchor_attn.src.modules.llama.anchor_attention import anchor_attention_forward  # noqa: E402
from anchor_attn.src.ops.anchor_attn_v4 import anchor_attn, dense_causal_attention  # noqa: E402
from anchor_attn.synthetic import stripe_positions  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
# (query heads, KV heads, head dimension, RoPE base)
LAYERS = {"llama8b": (32, 8, 128, 5e5), "qwen7b": (28, 4, 128, 1e6), "llama1b": (32, 8, 64, 5e5), "qwen05b": (14, 2, 64, 1e6)}
# (hidden size, MLP width): the models of the two Llama layer shapes
WIDTHS = {"llama8b": (4096, 14336), "llama1b": (2048, 8192)}
VOCAB = 32000
MODEL_LAYERS = 2


def _operator(layer, n, theta=12.0, regime="shared", dtype="bf16", block=128, step=16, batch=1):
    return {"kind": "operator", "layer": layer, "n": n, "theta": theta, "regime": regime, "dtype": dtype, "block": block,
            "step": step, "batch": batch}


def _plug(kind, layer, n, dtype="bf16", batch=1):
    return {"kind": kind, "layer": layer, "n": n, "dtype": dtype, "batch": batch}


def listed():
    return [
        # the headline: one Llama-3.1-8B layer at 128k tokens, about 0.6 % of the keys selected
        {"name": "operator_llama8b_128k", **_operator("llama8b", 131072)},
        # a group of seven query heads per KV head, 64k tokens
        {"name": "operator_qwen7b_64k", **_operator("qwen7b", 65536)},
        # the regime in which nearly every key passes the difference test: the sparse stage does the work of dense attention
        {"name": "operator_llama8b_32k_dense_regime", **_operator("llama8b", 32768, regime="literal")},
        # head dimension 64, fp16, smaller blocks (big blocks of 2048 keys from 64 x 32), a lower threshold
        {"name": "operator_llama1b_16k_fp16_block64", **_operator("llama1b", 16384, theta=11.0, dtype="fp16", block=64, step=32)},
        # a short context: two big blocks
        {"name": "operator_llama8b_4k", **_operator("llama8b", 4096)},
        # the smallest call: one big block of the smallest model, where launches and host time count
        {"name": "operator_qwen05b_2k", **_operator("qwen05b", 2048)},
        # a long prompt as it comes: nineteen big blocks and a tail of 1089 rows
        {"name": "prefill_llama8b_40001", **_plug("prefill", "llama8b", 40001)},
        # a short prompt, less than a big block
        {"name": "prefill_llama8b_777", **_plug("prefill", "llama8b", 777)},
        # one generated token against a 32k-token cache
        {"name": "decode_llama8b_33001", **_plug("decode", "llama8b", 33001)},
        # a batch of prompts of different lengths, padded on the left
        {"name": "padded_llama8b_3x2500", **_plug("padded", "llama8b", 2500, batch=3)},
        # the dense baseline
        {"name": "dense_llama8b_16k", **_plug("dense", "llama8b", 16384)},
        # a whole patched model's prefill
        {"name": "model_llama1b_6001", **_plug("model", "llama1b", 6001)},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["operator", "operator", "operator", "operator", "prefill", "prefill", "decode", "padded", "dense", "model"])
    layer = rng.choice(sorted(LAYERS))
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    if kind == "operator":
        block, step = rng.choice([(128, 16), (128, 16), (128, 16), (64, 16), (64, 32), (128, 32), (256, 16)])
        big = block * step
        regime = rng.choice(["shared", "shared", "shared", "literal"])
        n = max(1, _log_uniform(rng, 2048, 131072 if regime == "shared" else 24576) // big) * big
        theta = round(rng.uniform(10.0, 12.5), 1)
        batch = rng.choice([1, 1, 1, 2]) if n <= 32768 and regime == "shared" else 1
        return _operator(layer, n, theta, regime, dtype, block, step, batch)
    if kind == "prefill":
        n = _log_uniform(rng, 200, 40000)
        while (n % 2048) * n > 1089 * 40001:  # a tail no dearer than the listed one's
            n = _log_uniform(rng, 200, 40000)
        return _plug(kind, layer, n, dtype)
    if kind == "decode":
        batch = rng.choice([1, 1, 2, 4, 8])
        return _plug(kind, layer, _log_uniform(rng, 500, 131072 if batch == 1 else 40000), dtype, batch)
    if kind == "padded":
        batch = rng.choice([2, 3, 4])
        return _plug(kind, layer, _log_uniform(rng, 300, 3000 if batch == 4 else 4000), dtype, batch)
    if kind == "dense":
        return _plug(kind, layer, 128 * _log_uniform(rng, 4, 220), dtype)
    return _plug(kind, rng.choice(sorted(WIDTHS)), _log_uniform(rng, 300, 9000), "bf16")


# ---- inputs --------------------------------------------------------------------------------------------------------

def _qkv(layer, n, dtype, batch, seed, regime="shared", n_queries=None):
    """One layer's queries ``[B,Hq,N,D]`` (storage ``[B,N,Hq,D]``) and keys/values ``[B,Hkv,N,D]``; with ``n_queries`` only
    the last that many query rows."""
    hq, hkv, d, base = LAYERS[layer]
    dev, group = "cuda", hq // hkv
    gen = torch.Generator(device=dev).manual_seed(seed)
    host = torch.Generator().manual_seed(seed)
    inv = 1.0 / (base ** (torch.arange(0, d, 2, dtype=torch.float64, device=dev) / d))
    ang = torch.arange(n, dtype=torch.float64, device=dev)[:, None] * inv[None, :]
    cos = torch.cat([ang.cos(), ang.cos()], -1).float()
    sin = torch.cat([ang.sin(), ang.sin()], -1).float()
    del ang

    def rope(x, rows):
        return x * cos[rows] + torch.cat([-x[..., d // 2:], x[..., : d // 2]], -1) * sin[rows]

    n_q = n if n_queries is None else n_queries
    q_rows, all_rows = slice(n - n_q, n), slice(0, n)
    q = torch.empty(batch, n_q, hq, d, dtype=DTYPES[dtype], device=dev).transpose(1, 2)
    k = torch.empty(batch, hkv, n, d, dtype=DTYPES[dtype], device=dev)
    v = torch.empty(batch, hkv, n, d, dtype=DTYPES[dtype], device=dev)
    # half a per cent of the keys are stripes, thinning out with the distance from the start
    pos = stripe_positions(n, max(4, n // 200), "powerlaw", host).to(dev)
    for b in range(batch):
        shared = torch.randn(hkv, d, generator=gen, device=dev)
        shared *= math.sqrt(4.0 * math.sqrt(d)) / shared.norm(dim=-1, keepdim=True)
        for h in range(hkv):
            x = rope(torch.randn(group, n_q, d, generator=gen, device=dev), q_rows)
            add = shared[h] if regime == "shared" else x.mean((0, 1))
            q[b, h * group:(h + 1) * group] = (x + add if regime == "shared" else x).to(q.dtype)
            y = rope(torch.randn(n, d, generator=gen, device=dev), all_rows)
            y[0] += 4.0 * add
            y[pos] += 2.0 * add
            k[b, h] = y.to(k.dtype)
            v[b, h] = torch.randn(n, d, generator=gen, device=dev).to(v.dtype)
    return q, k, v


def _left_padded_mask(n, batch, seed, device):
    """Causal mask ``[B,1,N,N]`` of a left-padded batch: one prompt fills the row, the others lack up to half of it."""
    host = torch.Generator().manual_seed(seed)
    pads = [0] + [int(torch.randint(1, max(2, n // 2), (1,), generator=host)) for _ in range(batch - 1)]
    pos = torch.arange(n, device=device)
    real = pos[None, :] >= torch.tensor(pads, device=device)[:, None]
    return (pos[None, :] <= pos[:, None])[None, None] & real[:, None, None, :]


def prepare(case, seed):
    kind, layer, n, dtype, batch = (case[x] for x in ("kind", "layer", "n", "dtype", "batch"))
    if kind == "model":
        return _prepare_model(case, seed)
    q, k, v = _qkv(layer, n, dtype, batch, seed, case.get("regime", "shared"), 1 if kind == "decode" else None)
    state = {"kind": kind, "q": q, "k": k, "v": v, "scale": LAYERS[layer][2] ** -0.5}
    if kind == "operator":
        # what the operator's own callers hold: [B,H,N,D] tensors
        state.update(q=q.contiguous(), block=case["block"], step=case["step"], theta=case["theta"])
    elif kind == "dense":
        state.update(q=q.contiguous())
    else:
        state["module"] = types.SimpleNamespace(config=types.SimpleNamespace(block_size_M=128, step=16, theta=12.0))
        mask = _left_padded_mask(n, batch, seed, "cuda") if batch > 1 else None
        state["mask"] = mask[:, :, -1:].contiguous() if kind == "decode" and mask is not None else mask
    return state


def _prepare_model(case, seed):
    from transformers import LlamaConfig, LlamaForCausalLM

    from anchor_attn import patch_model
    hq, hkv, d, base = LAYERS[case["layer"]]
    hidden, mlp = WIDTHS[case["layer"]]
    config = LlamaConfig(hidden_size=hidden, intermediate_size=mlp, num_hidden_layers=MODEL_LAYERS, num_attention_heads=hq,
                         num_key_value_heads=hkv, head_dim=d, vocab_size=VOCAB, max_position_embeddings=131072, rope_theta=base)
    with torch.random.fork_rng(devices=[0]), torch.device("cuda"):
        torch.manual_seed(seed)
        model = LlamaForCausalLM(config).to(DTYPES[case["dtype"]]).eval()
        tokens = torch.randint(0, VOCAB, (case["batch"], case["n"]))
    return {"kind": "model", "model": patch_model(model, "anchor_attn"), "tokens": tokens}


# ---- one pass ------------------------------------------------------------------------------------------------------

def run(state):
    kind = state["kind"]
    if kind == "model":
        with torch.no_grad():
            got = state["model"](state["tokens"])
        layers = [(layer.keys, layer.values) for layer in got.past_key_values.layers]
        return {"logits": got.logits, "cache": layers}
    q, k, v = state["q"], state["k"], state["v"]
    if kind == "operator":
        out, ratio = anchor_attn(q, k, v, block_size=state["block"], step=state["step"], difference=state["theta"])
        return {"out": out, "ratio": ratio}
    if kind == "dense":
        return dense_causal_attention(q, k, v)
    return anchor_attention_forward(state["module"], q, k, v, state["mask"], scaling=state["scale"])[0]


# ---- what a pass cannot do without ---------------------------------------------------------------------------------

def _operator_flops(n, hq, d, block, step, regime):
    """Scores and P.V of the window [0,S) + [bb*S, r], pooled queries x candidate keys, and the selected keys (the stripes
    of the shared regime, all candidates of the literal one)."""
    big = block * step
    n_bb = n // big
    pairs = big * (big + 1) // 2 + (n_bb - 1) * (big * big + big * (big + 1) // 2)
    flops = 4.0 * d * pairs
    for bb in range(1, n_bb):
        candidates = max(bb * big - 2 * block, 0)
        chosen = candidates if regime == "literal" else max(4, n // 200) * math.sqrt(candidates / n)
        flops += 2.0 * step * d * candidates + 4.0 * d * big * chosen
    return hq * flops


def work(case):
    kind, n, batch = case["kind"], case["n"], case["batch"]
    hq, hkv, d, _ = LAYERS[case["layer"]]
    tokens_bytes = 2.0 * d * n * batch * (2 * hq + 2 * hkv)  # q, out, k, v of 16-bit elements
    causal = 4.0 * d * hq * batch * (n * (n + 1) // 2)
    if kind == "operator":
        return {"bytes": tokens_bytes, "flops": batch * _operator_flops(n, hq, d, case["block"], case["step"], case["regime"])}
    if kind == "decode":
        return {"bytes": 2.0 * d * batch * (2 * n * hkv + 2 * hq), "flops": 4.0 * d * hq * batch * n}
    if kind == "dense":
        return {"bytes": tokens_bytes, "flops": causal}
    if kind == "padded":  # (prompts are three quarters of the longest on average, so about half of the pairs are visible)
        return {"bytes": tokens_bytes + 1.0 * batch * n * n, "flops": causal * 0.6}
    main = n - n % 2048
    tail = 4.0 * d * hq * (n * (n + 1) // 2 - main * (main + 1) // 2)
    # a random model's scores lie close together: every key is selected
    attention = tail + (_operator_flops(main, hq, d, 128, 16, "literal" if kind == "model" else "shared") if main else 0.0)
    if kind == "prefill":
        return {"bytes": tokens_bytes, "flops": attention}
    hidden, mlp = WIDTHS[case["layer"]]
    weights = MODEL_LAYERS * (2 * hidden * hq * d + 2 * hidden * hkv * d + 3 * hidden * mlp)
    return {"bytes": 2.0 * (weights + VOCAB * hidden + n * hidden) + MODEL_LAYERS * tokens_bytes,
            "flops": 2.0 * weights * n + 2.0 * VOCAB * hidden + MODEL_LAYERS * attention}


def tolerance(case):
    """Four times the largest difference seen between the kernels and attention computed in float32 (2.5e-3 in bf16,
    3.2e-4 in fp16 where every key counts; single values near zero in the sum of many differ by up to 0.07 and 0.01 of the
    root mean square).  A whole model rounds to bf16 after each of its own operations as well: the same model with its dense
    rows computed in float32 differs by 9e-3."""
    if case["kind"] == "model":
        return {"rel": 3e-2, "max": 0.3}
    return {"rel": 1.5e-3, "max": 0.05} if case["dtype"] == "fp16" else {"rel": 1e-2, "max": 0.3}
