"""What a program built on this framework has it do, as cases that can be timed and compared.

A case is one call (or one attention-layer forward) through the public entry points:

* ``prefill``   - ``Xattention_prefill`` over a prompt, or over the next chunk of a prompt whose earlier tokens sit in
  a KV cache (``cache`` > 0);
* ``estimate``  - ``xattn_estimate``: block scores and the block mask without the attention;
* ``decode``    - ``single_decode_with_kv_cache``: one new token against the cache;
* ``layer``     - ``forward_eval``, the forward of a Llama attention layer (projections, rotary embedding, cache, then
  prefill or decode), as ``patch_model`` binds it.

Shapes are those of the repository's workloads (``xattn/synthetic.py``): 32 query heads with 8 or 32 KV heads, 28 with
4, 24 with 24; head dimension 128, bf16; inputs come from the same generators.
"""
import math
import os
import sys
import types

import torch

_PKG = os.path.join(os.getcwd(), "x-attention_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

from xattn.src.Xattention import Xattention_prefill, xattn_estimate  # noqa: E402
from xattn.src.decode import single_decode_with_kv_cache  # noqa: E402
from xattn.src.load_llama import FastPrefillConfig, forward_eval  # noqa: E402
from xattn.synthetic import ROPE_BASE, Workload, make_inputs  # noqa: E402

HIDDEN = 4096           # width of the layer cases' model (32 heads x 128)
D = 128
TAU_SPREAD = 0.08       # profiled per-head thresholds lie within about this much below and above their mean


def listed():
    return [
        # a short ragged prompt: what every chat request starts with; launches and host time count
        dict(name="prompt_1k", op="prefill", q=1000, cache=0, heads=32, kv_heads=8, stride=16, tau=0.9, per_head=False, causal=True, tokens="text", chunk=0),
        # workload 0 in the operator's own data type: a short document, one KV head per query head
        dict(name="prompt_4k_mha", op="prefill", q=4096, cache=0, heads=32, kv_heads=32, stride=8, tau=0.9, per_head=False, causal=True, tokens="text", chunk=2048),
        # workload 1: a long document
        dict(name="prompt_32k", op="prefill", q=32768, cache=0, heads=32, kv_heads=8, stride=8, tau=0.9, per_head=False, causal=True, tokens="text", chunk=16384),
        # workload 2: the longest context, the benchmark's headline
        dict(name="prompt_128k", op="prefill", q=131072, cache=0, heads=32, kv_heads=8, stride=16, tau=0.9, per_head=False, causal=True, tokens="text", chunk=16384),
        # workload 3: video frames followed by text, denser lists
        dict(name="video_64k", op="prefill", q=65536, cache=0, heads=28, kv_heads=4, stride=16, tau=0.9, per_head=False, causal=True, tokens="video", chunk=0),
        # workload 4: a video-generation transformer's layer, no causal mask, ragged length, the most work of all
        dict(name="field_119k", op="prefill", q=119056, cache=0, heads=24, kv_heads=24, stride=8, tau=0.95, per_head=False, causal=False, tokens="field", chunk=0),
        # chunked prefill: a serving loop feeds a long prompt 2048 tokens at a time on top of the cache
        dict(name="chunk_2k_of_64k", op="prefill", q=2048, cache=63488, heads=32, kv_heads=8, stride=16, tau=0.9, per_head=False, causal=True, tokens="text", chunk=0),
        # scores and mask on their own (analysis, threshold studies), ragged
        dict(name="estimate_16k", op="estimate", q=15000, cache=0, heads=32, kv_heads=8, stride=8, tau=0.9, per_head=False, causal=True, tokens="text", chunk=2048),
        # a decode step early in a conversation and one at the end of a long document
        dict(name="decode_1k", op="decode", q=1, cache=1100, heads=32, kv_heads=8),
        dict(name="decode_100k", op="decode", q=1, cache=100003, heads=32, kv_heads=8),
        # the next user turn: a few hundred tokens on a cache of a few thousand, profiled per-head thresholds,
        # through the whole attention layer
        dict(name="layer_turn_500", op="layer", q=500, cache=8700, heads=32, kv_heads=8, stride=16, tau=0.9, per_head=True, causal=True, tokens="text", chunk=0),
        # one generated token through the whole attention layer
        dict(name="layer_decode_9k", op="layer", q=1, cache=9200, heads=32, kv_heads=8, stride=16, tau=0.9, per_head=True, causal=True, tokens="text", chunk=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["prompt", "prompt", "prompt", "chunk", "chunk", "video", "field", "estimate", "decode", "decode", "layer", "layer"])
    heads, kv_heads = rng.choice([(32, 8), (32, 8), (32, 32), (28, 4)])
    case = dict(op="prefill", q=0, cache=0, heads=heads, kv_heads=kv_heads, stride=rng.choice([8, 16, 16]),
                tau=rng.choice([0.8, 0.9, 0.9, 0.95]), per_head=rng.random() < 0.3, causal=True, tokens="text", chunk=0)
    if kind == "prompt":
        case["q"] = _log_int(rng, 200, 131072)
        case["chunk"] = rng.choice([0, 0, 2048, 16384])
    elif kind == "chunk":
        case["q"] = _log_int(rng, 64, 8192)
        case["cache"] = _log_int(rng, 1000, 120000)
    elif kind == "video":
        case.update(heads=28, kv_heads=4, tokens="video", q=_log_int(rng, 4000, 65536))
    elif kind == "field":
        case.update(heads=24, kv_heads=24, stride=8, tokens="field", causal=False, q=_log_int(rng, 4000, 65536))
    elif kind == "estimate":
        case.update(op="estimate", q=_log_int(rng, 500, 65536), chunk=rng.choice([2048, 16384]))
    elif kind == "decode":
        case = dict(op="decode", q=1, cache=_log_int(rng, 100, 131072), heads=heads, kv_heads=kv_heads)
    else:
        decode = rng.random() < 0.5
        case.update(op="layer", heads=32, kv_heads=8, q=1 if decode else _log_int(rng, 64, 16384), cache=_log_int(rng, 500, 65536))
    return case


def _workload(case, length):
    kind = {"text": "text", "video": "video+text", "field": "field+text"}[case["tokens"]]
    full = 119056 if case["tokens"] == "field" else 65536      # the lengths at which the generators have their full grid
    return Workload("case", full, case["heads"], case["kv_heads"], case["stride"], case["tau"], None, case["causal"], kind), length


def _threshold(case, gen):
    """One tau, or - as the threshold profiler's tables hold them - one per head, kept on the host."""
    if not case["per_head"]:
        return case["tau"]
    spread = torch.rand(case["heads"], generator=gen) * 2 - 1
    return (case["tau"] + spread * min(TAU_SPREAD, 0.5 * (1 - case["tau"]))).to(torch.float32)


class _Cache:
    """A preallocated KV cache of one layer, with the ``update`` a model's cache has."""

    def __init__(self, kv_heads, capacity, filled, device):
        self.k = torch.zeros(1, kv_heads, capacity, D, dtype=torch.bfloat16, device=device)
        self.v = torch.zeros_like(self.k)
        self.filled = filled

    def update(self, key_states, value_states, layer_idx, cache_kwargs=None):
        end = self.filled + key_states.shape[2]
        self.k[:, :, self.filled:end] = key_states
        self.v[:, :, self.filled:end] = value_states
        return self.k[:, :, :end], self.v[:, :, :end]


def _layer_state(case, seed, device):
    """A Llama-shaped attention layer with random weights whose queries and keys look like the text generator's:
    feature 0 of the hidden state is constant (as the large activations of trained models are), and through it every
    query and key of a KV group gets that group's shared direction."""
    gen = torch.Generator(device=device).manual_seed(seed)
    H, Hkv, q_len, past = case["heads"], case["kv_heads"], case["q"], case["cache"]

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device=device)

    coeff, basis = randn(Hkv, 8), randn(8, D)
    direction = 2.0 * (coeff @ basis) / math.sqrt(8.0)
    bias = 4.0
    mod = types.SimpleNamespace()
    for name, n in (("q_proj", H), ("k_proj", Hkv), ("v_proj", Hkv)):
        lin = torch.nn.Linear(HIDDEN, n * D, bias=False, device=device, dtype=torch.bfloat16).requires_grad_(False)
        w = randn(n * D, HIDDEN) / math.sqrt(HIDDEN)
        w[:, 0] = 0.0 if name == "v_proj" else direction.repeat_interleave(n // Hkv, 0).reshape(-1) / bias
        lin.weight.copy_(w)
        setattr(mod, name, lin)
    mod.o_proj = torch.nn.Linear(H * D, HIDDEN, bias=False, device=device, dtype=torch.bfloat16).requires_grad_(False)
    mod.o_proj.weight.copy_(randn(HIDDEN, H * D) / math.sqrt(H * D))
    mod.config = types.SimpleNamespace(num_attention_heads=H, num_key_value_heads=Hkv)
    mod.head_dim, mod.layer_idx = D, 0
    tau = _threshold(case, torch.Generator().manual_seed(seed))
    mod.fastprefillconfig = FastPrefillConfig(threshold=tau[None] if case["per_head"] else tau, stride=case["stride"])
    hidden = randn(1, q_len, HIDDEN)
    hidden[..., 0] = bias
    inv = ROPE_BASE ** (-torch.arange(0, D, 2, dtype=torch.float32, device=device) / D)
    ang = torch.arange(past + q_len, dtype=torch.float32, device=device)[:, None] * inv[None, :]
    ang = torch.cat([ang, ang], dim=-1)
    cos, sin = ang.cos(), ang.sin()
    cache = _Cache(Hkv, past + q_len, past, device)
    for g in range(Hkv):
        x = randn(past, D) + direction[g]
        rot = torch.cat([-x[:, D // 2:], x[:, : D // 2]], dim=-1)
        cache.k[0, g, :past] = x * cos[:past] + rot * sin[:past]
        cache.v[0, g, :past] = randn(past, D)
    pos = (cos[None, past:].to(torch.bfloat16), sin[None, past:].to(torch.bfloat16))
    return dict(op="layer", mod=mod, hidden=hidden.to(torch.bfloat16), pos=pos, cache=cache)


def prepare(case, seed):
    device = torch.device("cuda", torch.cuda.current_device())
    with torch.no_grad():
        if case["op"] == "layer":
            return _layer_state(case, seed, device)
        if case["op"] == "decode":
            gen = torch.Generator(device=device).manual_seed(seed)
            L, Hkv, H = case["cache"], case["kv_heads"], case["heads"]
            cap = -(-(L + 1) // 1024) * 1024      # the cache is allocated ahead; the step reads a view of what is filled
            k = torch.randn(Hkv, cap, D, generator=gen, device=device, dtype=torch.bfloat16)
            v = torch.randn(Hkv, cap, D, generator=gen, device=device, dtype=torch.bfloat16)
            q = torch.randn(H, D, generator=gen, device=device, dtype=torch.bfloat16)
            return dict(op="decode", q=q, k=k[:, :L], v=v[:, :L])
        w, length = _workload(case, case["q"] + case["cache"])
        q, k, v = make_inputs(w, device=device, seed=seed, L=length)
        q = q[:, :, case["cache"]:].contiguous()
        # values come straight from a projection: [tokens, heads, 128] in memory
        v = v.transpose(1, 2).contiguous().transpose(1, 2)
        tau = _threshold(case, torch.Generator().manual_seed(seed))
        return dict(op=case["op"], q=q, k=k, v=v, tau=tau, stride=case["stride"], causal=case["causal"], chunk=case["chunk"] or None)


def run(state):
    op = state["op"]
    with torch.no_grad():
        if op == "prefill":
            return Xattention_prefill(state["q"], state["k"], state["v"], state["stride"], norm=1, threshold=state["tau"],
                                      chunk_size=state["chunk"], causal=state["causal"])
        if op == "estimate":
            sums, mask = xattn_estimate(state["q"], state["k"], 128, state["stride"], threshold=state["tau"],
                                        chunk_size=state["chunk"], causal=state["causal"])
            return {"sums": sums, "mask": mask}
        if op == "decode":
            return single_decode_with_kv_cache(state["q"], state["k"], state["v"], kv_layout="HND")
        cache = state["cache"]
        out, _ = forward_eval(state["mod"], state["hidden"], position_embeddings=state["pos"], past_key_values=cache)
        new = state["hidden"].shape[1]
        return {"out": out, "k": cache.k[:, :, -new:], "v": cache.v[:, :, -new:]}


def _kept_blocks(case):
    """Key blocks a query block's list holds on average for the generators' inputs (measured on them over a dozen seeds,
    tau 0.9 / 0.95): text 3 at 4k keys, 10 at 32k, 30 at 128k, and - on top of a cache - about four times as many, the
    queries all being far from the start; video 60 % and field 95-99 % of the visible ones."""
    q, k = case["q"], case["q"] + case["cache"]
    visible = (case["cache"] + (q / 2 if case["causal"] else q)) / 128 + 0.5
    if case["tokens"] == "text":
        return min(visible, (4 if case["cache"] else 1) * 3.05 * max(1.0, k / 4096) ** 0.63)
    return visible * (0.6 if case["tokens"] == "video" else 0.95)


def _attention_work(case):
    H, Hkv, q, k = case["heads"], case["kv_heads"], case["q"], case["q"] + case["cache"]
    if case["op"] == "decode" or (case["op"] == "layer" and q == 1):
        return 2.0 * (2 * H * D + 2 * Hkv * k * D), 4.0 * H * k * D
    pairs = q * (case["cache"] + q / 2) if case["causal"] else float(q) * k
    flops = 2.0 * H * D * pairs / case["stride"]              # the antidiagonal scores
    if case["op"] == "estimate":
        nq, nk = -(-q // 128), -(-k // 128)
        return 2.0 * D * (H * q + Hkv * k) + 3.0 * H * nq * nk, flops
    flops += 4.0 * 128 * 128 * D * H * -(-q // 128) * _kept_blocks(case)
    return 2.0 * D * (2 * H * q + 2 * Hkv * k), flops


def work(case):
    nbytes, flops = _attention_work(case)
    if case["op"] == "layer":
        n_out = (case["heads"] + 2 * case["kv_heads"]) * D
        weights = HIDDEN * (n_out + case["heads"] * D)
        nbytes += 2.0 * (weights + 2 * case["q"] * HIDDEN)
        flops += 2.0 * case["q"] * weights
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # everything comes back in bf16; a key block whose mass meets tau to within rounding may be kept or not, which
    # moves single mask entries and, through them, rows of the output
    if case["op"] == "estimate":
        return {"rel": 1e-2, "differ": 1e-3}
    return {"rel": 1e-2}
