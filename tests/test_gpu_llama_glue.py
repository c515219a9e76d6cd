"""GPU: the Llama attention forward (prefill on XAttention, decode on the
cache kernel) inside a small random-weight Llama, against the stock attention
of the installed model code and, for the sparse prefill, against the oracle
fed with the very tensors the layers passed to the operator."""
import copy

import pytest
import torch

from helpers import OUT_MAX_ABS, OUT_MEAN_ABS, mask_mismatch_report
from oracle import xattn_oracle as O

pytestmark = pytest.mark.gpu

transformers = pytest.importorskip("transformers")


def _tiny_llama(seed=0):
    from transformers import LlamaConfig
    from transformers.models.llama.modeling_llama import LlamaForCausalLM

    torch.manual_seed(seed)
    cfg = LlamaConfig(
        vocab_size=512, hidden_size=512, intermediate_size=1024, num_hidden_layers=2, num_attention_heads=4,
        num_key_value_heads=2, head_dim=128, max_position_embeddings=16384, rope_theta=500000.0,
        attn_implementation="eager",
    )
    return LlamaForCausalLM(cfg).to(torch.bfloat16).cuda().eval()


def _rel(a, b):
    return ((a.float() - b.float()).abs().max() / b.float().abs().max()).item()


def test_full_metric_prefill_and_decode_match_stock_attention():
    from xattn.src.load_llama import FastPrefillConfig, patch_model

    stock = _tiny_llama()
    ours = patch_model(copy.deepcopy(stock), FastPrefillConfig(threshold=0.9, metric="full"))
    ids = torch.randint(0, 512, (1, 1500), generator=torch.Generator().manual_seed(1)).cuda()
    with torch.no_grad():
        a = stock(ids, use_cache=True)
        b = ours(ids, use_cache=True)
        assert _rel(b.logits, a.logits) < 3e-2
        nxt = a.logits[:, -1:].argmax(-1)
        for _ in range(3):   # three decode steps on each model's own cache
            a = stock(nxt, past_key_values=a.past_key_values, use_cache=True)
            b = ours(nxt, past_key_values=b.past_key_values, use_cache=True)
            assert b.logits.shape == a.logits.shape == (1, 1, 512)
            assert _rel(b.logits, a.logits) < 3e-2
            nxt = a.logits[:, -1:].argmax(-1)


@pytest.mark.parametrize("mode", [torch.no_grad, torch.inference_mode])
def test_static_cache_is_cut_to_its_filled_part(mode):
    from transformers import StaticCache
    from xattn.src.load_llama import FastPrefillConfig, patch_model

    stock = _tiny_llama(5)
    ours = patch_model(copy.deepcopy(stock), FastPrefillConfig(threshold=0.9, metric="full"))
    ids = torch.randint(0, 512, (1, 700), generator=torch.Generator().manual_seed(6)).cuda()
    with mode():
        a = stock(ids, use_cache=True)                              # growing cache
        cache = StaticCache(config=ours.config, max_cache_len=1024)
        b = ours(ids, past_key_values=cache, use_cache=True)        # preallocated cache, 1024 slots
        assert _rel(b.logits, a.logits) < 3e-2
        nxt = a.logits[:, -1:].argmax(-1)
        for _ in range(2):
            a = stock(nxt, past_key_values=a.past_key_values, use_cache=True)
            b = ours(nxt, past_key_values=cache, use_cache=True)
            assert _rel(b.logits, a.logits) < 3e-2
            nxt = a.logits[:, -1:].argmax(-1)


def test_xattn_metric_calls_match_oracle(monkeypatch):
    from xattn.src import load_llama
    from xattn.src.load_llama import FastPrefillConfig, patch_model

    calls = []
    real = load_llama.Xattention_prefill

    def spy(q, k, v, stride, **kw):
        out = real(q, k, v, stride, **kw)
        calls.append((q.detach().cpu(), k.detach().cpu(), v.detach().cpu(), stride, kw, out.detach().cpu()))
        return out

    monkeypatch.setattr(load_llama, "Xattention_prefill", spy)
    tau = torch.tensor([[0.9, 0.8, 0.95, 0.5], [1.0, 0.0, 0.9, 0.7]])
    model = patch_model(_tiny_llama(2), FastPrefillConfig(threshold=tau, stride=8))
    ids = torch.randint(0, 512, (1, 2100), generator=torch.Generator().manual_seed(3)).cuda()
    with torch.no_grad():
        first = model(ids[:, :1300], use_cache=True)                 # prefill
        model(ids[:, 1300:], past_key_values=first.past_key_values, use_cache=True)   # second chunk on the cache
    assert len(calls) == 4
    from xattn.src.Xattention import default_chunk_size, xattn_estimate

    for layer, (q, k, v, stride, kw, out) in zip([0, 1, 0, 1], calls):
        assert q.shape[1] == 4 and k.shape[1] == 2 and stride == 8      # KV heads not repeated
        assert (q.shape[2], k.shape[2]) in ((1300, 1300), (800, 2100))
        assert torch.equal(kw["threshold"].cpu(), tau[layer])
        # the layer's result is the operator's: oracle attention under the mask the
        # estimator selects for these very tensors (mask parity itself is covered
        # by the operator tests; here the same band check against the oracle's mask)
        chunk = default_chunk_size(k.shape[2])
        _, mask = xattn_estimate(q.cuda(), k.cuda(), 128, stride, threshold=kw["threshold"], chunk_size=chunk)
        nq, nk = (q.shape[2] + 127) // 128, (k.shape[2] + 127) // 128
        want_sums, want_mask = O.xattn_estimate(
            q.float(), k.repeat_interleave(2, 1).float(), 128, stride, threshold=kw["threshold"].cpu(),
            chunk_size=chunk, pad0_quirk=False,
        )
        nbad, outside = mask_mismatch_report(want_sums[0], mask[0], want_mask[0], kw["threshold"].cpu(), True,
                                             mask.shape[3] - mask.shape[2], chunk // 128)
        assert outside == 0, (layer, nbad, outside)
        mask = mask[:, :, :nq, :nk].cpu()
        want = O.block_sparse_attention(q, k, v, mask, causal=True)
        err = (out.float() - want.float()).abs()
        assert err.max().item() <= OUT_MAX_ABS and err.mean().item() <= OUT_MEAN_ABS


def test_a_replaced_decode_call_sees_every_step(monkeypatch):
    """A program that puts its own function in the decode call's place, as the prefill's above, gets each layer's step, with
    the arguments of the call and its result used; the result is that of the ordinary step to the bit."""
    from xattn.src import load_llama
    from xattn.src.load_llama import FastPrefillConfig, patch_model

    model = patch_model(_tiny_llama(7), FastPrefillConfig(threshold=0.9))
    ids = torch.randint(0, 512, (1, 301), generator=torch.Generator().manual_seed(8)).cuda()
    real, calls = load_llama.single_decode_with_kv_cache, []

    def step():
        with torch.no_grad():
            first = model(ids[:, :300], use_cache=True)
            return model(ids[:, 300:], past_key_values=first.past_key_values, use_cache=True).logits

    def spy(q, k, v, **kw):
        calls.append((q.shape, k.shape, v.shape, kw))
        return real(q, k, v, **kw)

    want = step()
    monkeypatch.setattr(load_llama, "single_decode_with_kv_cache", spy)
    assert torch.equal(step(), want)
    assert calls == [((4, 128), (2, 301, 128), (2, 301, 128), {"kv_layout": "HND"})] * 2
    monkeypatch.setattr(load_llama, "single_decode_with_kv_cache", lambda q, k, v, **kw: torch.zeros_like(q))
    assert not torch.equal(step(), want)


def test_batch_two_is_refused():
    from xattn.src.load_llama import FastPrefillConfig, patch_model

    model = patch_model(_tiny_llama(4), FastPrefillConfig(threshold=0.9))
    with pytest.raises(ValueError), torch.no_grad():
        model(torch.zeros(2, 256, dtype=torch.long, device="cuda"))
