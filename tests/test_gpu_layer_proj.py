"""GPU: the projection and rotation kernels of the attention layer (through the native host path) against the torch
expressions they stand for."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(x, weights, biases, heads, cos, sin):
    """q, k, v as the reference's layer computes them, the products in fp32 and rounded once."""
    from xattn.src.load_llama import apply_rotary_pos_emb

    out = []
    for w, b, n in zip(weights, biases, heads):
        y = x.float() @ w.float().t() + (b.float() if b is not None else 0.0)
        out.append(y.bfloat16().view(1, x.shape[1], n, 128).transpose(1, 2))
    out[0], out[1] = apply_rotary_pos_emb(out[0], out[1], cos, sin)
    return out


# widths around the loads of a row: less than one chunk of 512, chunk and batch (2048) edges, an odd number of batches
@pytest.mark.parametrize("width", [8, 504, 512, 520, 2048, 2056, 6144])
@pytest.mark.parametrize("tokens,heads,kv_heads,bias", [(1, 4, 1, True), (1, 6, 6, False), (2, 4, 2, True), (77, 3, 1, False)])
def test_projection_and_rotation(width, tokens, heads, kv_heads, bias):
    from xattn.src import hip_backend as hb

    g = torch.Generator(device="cuda").manual_seed(width + tokens)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    n = (heads, kv_heads, kv_heads)
    weights = [(rnd(h * 128, width) / width ** 0.5).bfloat16() for h in n]
    biases = [rnd(h * 128).bfloat16() if bias else None for h in n]
    x = rnd(1, tokens, width).bfloat16()
    ang = rnd(1, tokens, 128) * 3
    cos, sin = ang.cos().bfloat16(), ang.sin().bfloat16()
    with torch.no_grad():
        got = hb.host().project(x, weights[0], biases[0], weights[1], biases[1], weights[2], biases[2], cos, sin, heads, kv_heads)
        want = _reference(x, weights, biases, n, cos, sin)
        # fp32 sums in another order: a result next to a rounding boundary may land one bf16 step (2^-8 of its
        # magnitude) away; the rotation adds two such values and rounds once more
        for a, b in zip(got, want):
            assert a.shape == b.shape
            assert ((a.float() - b.float()).abs() <= 3 * 2.0 ** -8 * (b.float().abs() + 1)).all()
            assert (a != b).float().mean() < 0.02
        if tokens == 1:
            y = hb.host().output(x, weights[0], biases[0])
            ref = (x.float() @ weights[0].float().t() + (biases[0].float() if bias else 0.0)).bfloat16()
            assert ((y.float() - ref.float()).abs() <= 2.0 ** -8 * (ref.float().abs() + 1)).all()


# one token: a wavefront's share of a row (every fourth chunk of 512) of one, two, four and more chunks and the first width beyond each,
# some wavefronts without any; weights around 24 MiB, from which they are loaded not temporal
@pytest.mark.parametrize("width,heads,kv_heads", [(16, 1, 1), (1544, 2, 1), (4096, 4, 2), (4104, 4, 2), (8192, 2, 2), (8200, 2, 1), (10248, 3, 1),
                                                  (24576, 2, 1), (2048, 32, 8), (2048, 32, 9)])
def test_one_token(width, heads, kv_heads):
    test_projection_and_rotation(width, 1, heads, kv_heads, width % 16 == 0)


def test_one_token_and_more_rows_than_a_launch_has():
    from xattn.src import hip_backend as hb

    n = (1 << 24) + 4
    g = torch.Generator(device="cuda").manual_seed(0)
    w = torch.randn(n, 8, generator=g, device="cuda", dtype=torch.bfloat16)
    b = torch.randn(n, generator=g, device="cuda", dtype=torch.bfloat16)
    x = torch.randn(1, 1, 8, generator=g, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        y = hb.host().output(x, w, b)
        ref = (w.float() * x.float()[0]).sum(-1) + b.float()
    assert ((y[0, 0].float() - ref).abs() <= 2.0 ** -8 * (ref.abs() + 1)).all()


def test_modules_that_are_more_than_a_linear_are_called():
    """A hook or a replaced forward on a projection means that the module itself runs."""
    from xattn.src.load_llama import _linear_params

    lin = torch.nn.Linear(512, 512, bias=False)
    assert _linear_params(lin) is not None
    handle = lin.register_forward_hook(lambda *a: None)
    assert _linear_params(lin) is None
    handle.remove()
    lin.forward = lambda x: x
    assert _linear_params(lin) is None
    assert _linear_params(torch.nn.Identity()) is None


def test_a_linear_replaced_on_the_class_is_called(monkeypatch):
    """A wrapper around torch.nn.Linear.forward, or a mode, sees the layer's four products."""
    import types

    from xattn.src.load_llama import FastPrefillConfig, forward_eval

    heads, kv_heads, width, tokens = 4, 2, 256, 70
    g = torch.Generator(device="cuda").manual_seed(0)
    mod = types.SimpleNamespace(config=types.SimpleNamespace(num_attention_heads=heads, num_key_value_heads=kv_heads), head_dim=128,
                                layer_idx=0, fastprefillconfig=FastPrefillConfig(threshold=0.9))
    for name, n, k in (("q_proj", heads * 128, width), ("k_proj", kv_heads * 128, width), ("v_proj", kv_heads * 128, width),
                       ("o_proj", width, heads * 128)):
        lin = torch.nn.Linear(k, n, bias=False, device="cuda", dtype=torch.bfloat16).requires_grad_(False)
        lin.weight.copy_(torch.randn(n, k, generator=g, device="cuda") / k ** 0.5)
        setattr(mod, name, lin)
    x = torch.randn(1, tokens, width, generator=g, device="cuda").bfloat16()
    ang = torch.rand(1, tokens, 128, generator=g, device="cuda") * 3
    pos = (ang.cos().bfloat16(), ang.sin().bfloat16())
    plain = torch.nn.Linear.forward
    calls = []

    def forward(self, a):
        calls.append(tuple(self.weight.shape))
        return plain(self, a)

    with torch.no_grad():
        want = forward_eval(mod, x, position_embeddings=pos)[0]
        assert not calls
        monkeypatch.setattr(torch.nn.Linear, "forward", forward)
        got = forward_eval(mod, x, position_embeddings=pos)[0]
        assert len(calls) == 4
        monkeypatch.undo()
        seen = []

        class Mode(torch.overrides.TorchFunctionMode):
            def __torch_function__(self, func, types, args=(), kwargs=None):
                seen.append(func)
                return func(*args, **(kwargs or {}))

        with Mode():
            forward_eval(mod, x, position_embeddings=pos)
        assert seen.count(torch.nn.functional.linear) == 4
    # products rounded to bf16 by both, their sums in another order, through a softmax and one more product
    assert (got.float() - want.float()).norm() <= 2e-2 * want.float().norm()
