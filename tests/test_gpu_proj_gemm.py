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
    # 128 x 128, and tiles of 192 and 256 tokens
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


# CUs without a tile pull weights ahead, from the sixth step on (64 x 64) or the fourth: few tiles, none but one XCD's at work, runs of
# tiles that end inside a head, last token tiles with enough rows for it and with too few; then tiles of 192 and 256 tokens, whole
# and with a remainder, steps odd and even
@pytest.mark.parametrize("tokens,heads,kv_heads,width", [
    (40, 1, 1, 4096), (2, 3, 1, 1088), (150, 5, 3, 2048), (115, 5, 3, 2048), (191, 32, 8, 448), (500, 28, 4, 1024), (250, 32, 8, 704), (600, 32, 8, 4160),
    (769, 32, 8, 576), (960, 32, 8, 512), (1025, 32, 8, 640), (1280, 32, 8, 832),
])
def test_weights_pulled_ahead_and_large_tiles(tokens, heads, kv_heads, width):
    test_projections_of_a_turn(tokens, heads, kv_heads, width, True)


@pytest.mark.parametrize("width", [64, 128, 192, 256, 320, 384, 448])
@pytest.mark.parametrize("tokens", [5, 200, 320, 500, 640, 700, 1000])
def test_depths_of_a_few_slabs(tokens, width):
    """One slab to one more than the deepest ring of stages holds, with every tile."""
    test_projections_of_a_turn(tokens, 32, 8, width, True)


def test_two_workgroups_per_cu():
    """2600 tokens of 24 heads: 504 tiles of 128 x 128, but more than 256 of 256 tokens."""
    from xattn.src import hip_backend as hb

    g = torch.Generator(device="cuda").manual_seed(2600)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    assert hb.lib().xattn_proj_gemm_fits(2600, 448, 24 * 128, 1)
    weights = [(rnd(h * 128, 448) / 448 ** 0.5).bfloat16() for h in (16, 4, 4)]
    x, cos, sin = rnd(1, 2600, 448).bfloat16(), torch.ones(1, 2600, 128, device="cuda").bfloat16(), torch.zeros(1, 2600, 128, device="cuda").bfloat16()
    with torch.no_grad():
        got = hb.host().project(x, weights[0], None, weights[1], None, weights[2], None, cos, sin, 16, 4)
        for a, b in zip(got, _reference(x, weights, (None,) * 3, (16, 4, 4), cos, sin)):
            # one bf16 step where the fp32 sums, in another order, round to the other side (nothing is rotated)
            assert ((a.float() - b.float()).abs() <= 2.0 ** -7 * b.float().abs() + 1e-5).all() and (a != b).float().mean() < 0.02


@pytest.mark.parametrize("tokens,heads,taken", [(1100, 32, True), (1536, 32, True), (1537, 32, False), (640, 64, True)])
def test_output_of_many_tokens(tokens, heads, taken):
    from xattn.src import hip_backend as hb

    g = torch.Generator(device="cuda").manual_seed(tokens)
    x = torch.randn(1, tokens, 704, generator=g, device="cuda").bfloat16()
    w = (torch.randn(heads * 128, 704, generator=g, device="cuda") / 704 ** 0.5).bfloat16()
    with torch.no_grad():
        y = hb.host().output(x, w, None)
    assert (y is not None) == taken
    if taken:
        ref = (x.float() @ w.float().t()).bfloat16()
        # one bf16 step where the fp32 sums, in another order, round to the other side
        assert ((y.float() - ref.float()).abs() <= 2.0 ** -7 * ref.float().abs() + 1e-5).all() and (y != ref).float().mean() < 0.02
