"""GPU: the projections of a turn of some hundred tokens as one kernel, against products in fp32 rounded once."""
import pytest
import torch

from test_gpu_layer_proj import _reference

pytestmark = pytest.mark.gpu

SIZES = [
    # 64 x 64 tiles: one token in a tile, its edges; fewer steps than stages, as many, one more
    (2, 1, 1, 64), (63, 4, 2, 128), (64, 4, 1, 320), (65, 4, 4, 384), (77, 3, 1, 448), (128, 32, 8, 64),
    # 64 tokens x 128 features
    (129, 32, 8, 128), (320, 32, 8, 192), (193, 28, 4, 320),
    # 128 x 128, four stages and two
    (321, 32, 8, 256), (640, 32, 8, 64), (641, 32, 8, 128), (1280, 32, 8, 192), (900, 32, 8, 64),
    # the library's
    (1281, 32, 8, 64), (77, 4, 2, 72),
]


@pytest.mark.parametrize("tokens,heads,kv_heads,width", SIZES)
@pytest.mark.parametrize("bias", [True, False])
def test_projections_of_a_turn(tokens, heads, kv_heads, width, bias):
    from xattn.src import hip_backend as hb

    g = torch.Generator(device="cuda").manual_seed(width + tokens)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    n = (heads, kv_heads, kv_heads)
    # weights whose rows lie further apart than they are long, as slices of a fused matrix do
    weights = [(rnd(h * 128, width + 8) / width ** 0.5).bfloat16()[:, :width] for h in n]
    biases = [rnd(h * 128).bfloat16() if bias else None for h in n]
    x = rnd(1, tokens, width).bfloat16()
    ang = rnd(1, tokens, 128) * 3
    cos, sin = ang.cos().bfloat16(), ang.sin().bfloat16()
    lib = hb.lib()
    assert lib.xattn_proj_gemm_fits(tokens, width, sum(n) * 128, 1) == (tokens < 1281 and width % 64 == 0)
    with torch.no_grad():
        got = hb.host().project(x, weights[0], biases[0], weights[1], biases[1], weights[2], biases[2], cos, sin, heads, kv_heads)
        want = _reference(x, weights, biases, n, cos, sin)
        # fp32 sums in another order: a result next to a rounding boundary may land one bf16 step away, at most 2^-7 of its
        # magnitude.  The rotation adds two such values, each times at most 1, and its three roundings of 2^-9 each may fall to
        # the other side: twice a step of each covers them.
        close = lambda a, b, size: ((a.float() - b.float()).abs() <= size + 1e-5).all() and (a != b).float().mean() < 0.02
        plain = _reference(x, weights, biases, n, torch.ones_like(cos), torch.zeros_like(sin))
        for a, b, u in zip(got[:2], want[:2], plain[:2]):
            assert a.shape == b.shape
            assert close(a, b, 2 * 2.0 ** -7 * (u.float().abs() + u.float().abs().roll(64, -1)))
        assert close(got[2], want[2], 2.0 ** -7 * want[2].float().abs())
        y = hb.host().output(x, weights[0], biases[0])
        assert (y is not None) == bool(lib.xattn_proj_gemm_fits(tokens, width, heads * 128, 0))
        if y is not None:
            ref = (x.float() @ weights[0].float().t() + (biases[0].float() if bias else 0.0)).bfloat16()
            assert close(y, ref, 2.0 ** -7 * ref.float().abs())
