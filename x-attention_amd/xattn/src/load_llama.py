"""Llama attention forward on the HIP prefill and decode kernels.

Mirror of xattn/src/load_llama.py of mit-han-lab/x-attention: the same
``FastPrefillConfig`` / ``forward_eval`` / ``load_model`` names, with three
differences that the kernels make possible:

* K and V keep their ``H_kv`` heads - the reference repeats them to ``H`` heads
  before the operator (``repeat_kv``, load_llama.py:158-159), the kernels share
  a KV head among its query heads instead;
* the decode step (one new token against the cache) runs on
  :func:`xattn.src.decode.single_decode_with_kv_cache` where the reference
  calls flashinfer (load_llama.py:180-197);
* ``metric="full"`` is the same attention kernel visiting every visible block
  (the reference calls flash-attn, xattn/src/Fullprefill.py).

``metric="flex"`` and ``metric="minfer"`` are other sparse-attention methods the
reference carries for comparison; they are not provided here.
"""
import inspect
import sys
import time

import torch
import torch.autograd.forward_ad
import torch.utils._device

from . import hip_backend as _hb
from .decode import single_decode_with_kv_cache
from .Xattention import Xattention_prefill, block_sparse_attention

__all__ = ["FastPrefillConfig", "forward_eval", "patch_model", "load_model", "apply_rotary_pos_emb", "rotate_half"]


def rotate_half(x):
    half = x.shape[-1] // 2
    return torch.cat((-x[..., half:], x[..., :half]), dim=-1)


def apply_rotary_pos_emb(q, k, cos, sin, unsqueeze_dim=1):
    """Rotate-half rotary embedding on ``[B, H, L, d]`` tensors (load_llama.py:41-65)."""
    cos, sin = cos.unsqueeze(unsqueeze_dim), sin.unsqueeze(unsqueeze_dim)
    return q * cos + rotate_half(q) * sin, k * cos + rotate_half(k) * sin


class FastPrefillConfig(dict):
    """Settings of the prefill path (load_llama.py:224-259).

    threshold:  float - one tau for every layer and head;
                tensor ``[layers, heads]`` - per-layer rows of per-head taus, as
                produced by the threshold profiler;
                None - the profiled table of this stride,
                ``xattn.threshold.llama_threshold.llama_fuse_<stride>``
                (``[layers][heads]``; load_llama.py:254-261).  That module reads
                the tables from a JSON file the profiler writes, or can be
                replaced by the reference's own module of the same name (tables
                profiled on Llama-3.1-8B-Instruct, parameters of that model,
                not shipped here); without either it raises ``ValueError``.
    stride:     antidiagonal stride, 4, 8 or 16.
    metric:     "xattn" or "full".
    print_detail: print per-stage wall times (synchronises the device).
    """

    def __init__(self, threshold=None, print_detail=False, stride=16, metric="xattn"):
        super().__init__()
        if stride not in (4, 8, 16):
            raise ValueError("stride must be 4, 8 or 16")
        if metric not in ("xattn", "full"):
            raise NotImplementedError(f"metric {metric!r}: only 'xattn' and 'full' are provided")
        self.print_detail = print_detail
        self.metric = metric
        self.stride = stride
        if threshold is None:
            # the profiled [layers, heads] table of this stride (xattn/src/load_llama.py:254-261);
            # raises ValueError naming where a table is looked for when there is none
            from xattn.threshold import llama_threshold as tables

            threshold = torch.tensor(getattr(tables, f"llama_fuse_{stride}"), dtype=torch.float32)
        if isinstance(threshold, torch.Tensor):
            if threshold.dim() != 2:
                raise ValueError("a threshold tensor must be [layers, heads]")
            self.threshold = threshold.detach().to(torch.float32)
        else:
            self.threshold = float(threshold)

    def layer_threshold(self, layer_idx):
        """tau of one layer: a float or a ``[heads]`` tensor."""
        if isinstance(self.threshold, torch.Tensor):
            return self.threshold[layer_idx]
        return self.threshold


def _is_static_cache(cache):
    if "transformers" not in sys.modules:      # then nobody holds one
        return False
    try:
        from transformers import StaticCache
    except ImportError:
        return False
    return isinstance(cache, StaticCache)


_module_hooks = torch.nn.modules.module


def _torch_own(fn, module):
    """Whether a function comes from the file of a torch module, as it does unless something has replaced it."""
    code = getattr(fn, "__code__", None)
    return code is not None and code.co_filename == module.__file__


_Linear, _functional = torch.nn.Linear, torch.nn.functional


def _linear_call():
    """What a call of a ``torch.nn.Linear`` goes through."""
    return _Linear.__call__, _Linear._call_impl, _Linear.forward, _functional.linear


_own_linear_call = _linear_call()
if not (all(_torch_own(fn, _module_hooks) for fn in _own_linear_call[:2])
        and _torch_own(_own_linear_call[2], torch.nn.modules.linear) and _own_linear_call[3] is torch._C._nn.linear):
    _own_linear_call = None      # replaced before this module was imported
_own_decode = single_decode_with_kv_cache
_function_modes, _dispatch_modes = torch._C._len_torch_function_stack, torch._C._len_torch_dispatch_stack
_forward_ad, _transform, _tracer = torch.autograd.forward_ad, torch._C._functorch.peek_interpreter_stack, torch._C._get_tracing_state


def _observed():
    """Whether something wants to see the calls that torch functions and modules make: a function or dispatch mode
    (other than a default device, which only concerns new tensors), forward-mode differentiation, a functorch transform, a
    tracer, or a replaced part of ``torch.nn.Linear``'s call."""
    if _linear_call() != _own_linear_call:
        return True
    if _function_modes() and any(type(m) is not torch.utils._device.DeviceContext
                                 for m in torch.overrides._get_current_function_mode_stack()):
        return True
    return bool(_dispatch_modes()) or _forward_ad._current_level >= 0 or _transform() is not None or _tracer() is not None


def _linear_params(mod):
    """(weight, bias) of a projection that is nothing but ``torch.nn.Linear`` - no hooks, no replaced forward, not
    compiled, no wrapped or quantized weight - so that its product may be computed without calling the module where
    nothing observes the call; else None."""
    own = mod.__dict__
    if (type(mod) is not torch.nn.Linear or "forward" in own or own["_forward_hooks"] or own["_forward_pre_hooks"]
            or own.get("_compiled_call_impl") is not None
            or _module_hooks._global_forward_hooks or _module_hooks._global_forward_pre_hooks):
        return None
    weight, bias = own["_parameters"].get("weight"), own["_parameters"].get("bias")
    if type(weight) is not torch.nn.Parameter or (bias is not None and type(bias) is not torch.nn.Parameter):
        return None
    return weight, bias


def _project(self, hidden_states, cos, sin, heads, kv_heads):
    """Rotated q and k and v of a layer from the native host path (one kernel up to about a thousand tokens, the library
    GEMMs and one rotation kernel for more), or None where the layer's own modules have to be called."""
    if self.head_dim != 128:
        return None
    q, k, v = _linear_params(self.q_proj), _linear_params(self.k_proj), _linear_params(self.v_proj)
    if q is None or k is None or v is None:
        return None
    return _hb.host().project(hidden_states, *q, *k, *v, cos, sin, heads, kv_heads)


def _stamp(cfg, label, start):
    if cfg.print_detail:
        torch.cuda.synchronize()
        print(f"     {label} took: {time.time() - start:.6f} seconds")
    return time.time()


def forward_eval(self, hidden_states, position_embeddings=None, attention_mask=None, past_key_values=None,
                 past_key_value=None, cache_position=None, position_ids=None, **kwargs):
    """Attention layer forward, prefill on XAttention and decode on the cache
    kernel (load_llama.py:80-220).  Bound to every ``self_attn`` by
    :func:`patch_model`; ``self.fastprefillconfig`` carries the settings.

    Batch size must be 1 (the operator's own limit, Xattention.py:357).  A
    call with one query token and a longer cache is a decode step; everything
    else (first prefill, or a further chunk of a chunked prefill on top of the
    cache) goes through the prefill operator, whose causal mask is aligned to
    the end of the cache.
    """
    cfg = self.fastprefillconfig
    start = time.time()
    bsz, q_len, _ = hidden_states.size()
    if bsz != 1:
        raise ValueError("the XAttention forward handles batch size 1")
    heads = self.config.num_attention_heads
    kv_heads = self.config.num_key_value_heads
    head_dim = self.head_dim

    native = hidden_states.is_cuda and type(hidden_states) is torch.Tensor and not _observed()
    qkv = None
    if position_embeddings is not None:
        cos, sin = position_embeddings
    if position_embeddings is not None and native:
        qkv = _project(self, hidden_states, cos, sin, heads, kv_heads)
    if qkv is not None:
        query_states, key_states, value_states = qkv
        start = _stamp(cfg, "Reshape", start)
    else:
        query_states = self.q_proj(hidden_states).view(bsz, q_len, heads, head_dim).transpose(1, 2)
        key_states = self.k_proj(hidden_states).view(bsz, q_len, kv_heads, head_dim).transpose(1, 2)
        value_states = self.v_proj(hidden_states).view(bsz, q_len, kv_heads, head_dim).transpose(1, 2)
        start = _stamp(cfg, "Reshape", start)
        if position_embeddings is None:
            cos, sin = self.rotary_emb(value_states, position_ids)
        query_states, key_states = apply_rotary_pos_emb(query_states, key_states, cos, sin)

    cache = past_key_values if past_key_values is not None else past_key_value
    if cache is not None:
        cache_kwargs = {"sin": sin, "cos": cos, "cache_position": cache_position}
        key_states, value_states = cache.update(key_states, value_states, self.layer_idx, cache_kwargs)
        if _is_static_cache(cache):
            # a preallocated cache hands back its whole buffer: keep what is filled (load_llama.py:152-154).
            # The last position comes from cache_position where the model code passes it, else from position_ids.
            pos = cache_position if cache_position is not None else (position_ids[0] if position_ids is not None else None)
            if pos is None:
                raise ValueError("a static cache needs cache_position or position_ids to know how much of it is filled")
            # reading the position costs a device-to-host copy: the first layer of a model forward does it, the
            # other layers (handed the same positions) reuse its value.  Nothing here depends on tensor
            # identity or version counters, which inference-mode tensors do not have.
            memo = getattr(cfg, "_filled_memo", None)
            if memo is None or self.layer_idx in (0, None):
                last = int(pos[-1])
                cfg._filled_memo = (last,)
            else:
                last = memo[0]
            filled = min(last + 1, key_states.shape[2])
            key_states, value_states = key_states[:, :, :filled], value_states[:, :, :filled]
    if key_states.device != query_states.device:
        key_states = key_states.to(query_states.device)
        value_states = value_states.to(query_states.device)
    k_len = key_states.shape[2]
    decoding = q_len != k_len and q_len == 1
    start = _stamp(cfg, "Past KV update", start)
    if cfg.print_detail:
        print(f"q length: {q_len} k length: {k_len}")

    # the ordinary decode step comes back as the output projection takes it, without views made and put together here (not where a
    # program has put a function of its own in this module's decode call)
    merged = None
    if decoding and native and single_decode_with_kv_cache is _own_decode and type(query_states) is type(key_states) is type(value_states) is torch.Tensor:
        merged = _hb.host().decode_layer(query_states, key_states, value_states)
    if merged is not None:
        pass
    elif decoding:
        attn_output = single_decode_with_kv_cache(
            query_states[0, :, 0], key_states[0], value_states[0], kv_layout="HND"
        ).reshape(1, heads, 1, head_dim)
    elif cfg.metric == "xattn":
        threshold = cfg.layer_threshold(self.layer_idx)
        attn_output = Xattention_prefill(
            query_states, key_states, value_states, cfg.stride, norm=1, threshold=threshold, use_triton=True
        )
    else:
        attn_output = block_sparse_attention(query_states, key_states, value_states, causal=True)
    start = _stamp(cfg, "Attention computation", start)

    if merged is not None:
        attn_output = merged
    else:
        if attn_output.size() != (bsz, heads, q_len, head_dim):
            raise ValueError(
                f"`attn_output` should be of size {(bsz, heads, q_len, head_dim)}, but is {attn_output.size()}"
            )
        attn_output = attn_output.transpose(1, 2).reshape(bsz, q_len, heads * head_dim)
    out_proj = _linear_params(self.o_proj) if native else None
    projected = _hb.host().output(attn_output, *out_proj) if out_proj is not None else None
    attn_output = projected if projected is not None else self.o_proj(attn_output)
    _stamp(cfg, "Post-attention processing", start)
    if getattr(self, "_xattn_three_outputs", False):
        return attn_output, None, cache
    return attn_output, None


def patch_model(model, fastprefillconfig):
    """Binds :func:`forward_eval` to every attention layer of a Llama model that
    is already in memory (what load_llama.py:283-285 does after loading)."""
    for layer in model.model.layers:
        attn = layer.self_attn
        if attn.head_dim != 128:
            raise ValueError("the kernels are built for head_dim 128")
        # older releases of the model code unpack three values from the layer's forward
        attn._xattn_three_outputs = "past_key_values" not in inspect.signature(type(attn).forward).parameters
        attn.fastprefillconfig = fastprefillconfig
        attn.forward = forward_eval.__get__(attn)
    return model


def load_model(fastprefillconfig=None, name_or_path=""):
    """Loads a Llama checkpoint in bf16 on the GPU and patches its attention
    (load_llama.py:261-290).  Returns ``(model, tokenizer)``."""
    from transformers import AutoTokenizer
    from transformers.models.llama.modeling_llama import LlamaForCausalLM

    if fastprefillconfig is None:
        fastprefillconfig = FastPrefillConfig()
    model = LlamaForCausalLM.from_pretrained(name_or_path, device_map="cuda", torch_dtype=torch.bfloat16)
    model.eval()
    patch_model(model, fastprefillconfig)
    return model, AutoTokenizer.from_pretrained(name_or_path)
