"""GPU parity: xattn_decode_fwd (through the C ABI) vs the CPU oracle."""
import pytest
import torch

from helpers import OUT_MAX_ABS, OUT_MEAN_ABS
from oracle import xattn_oracle as O

pytestmark = pytest.mark.gpu


def _mk(H, Hkv, L, seed, spread=1.0):
    g = torch.Generator().manual_seed(seed)
    q = (torch.randn(H, 128, generator=g) * spread).bfloat16()
    k = torch.randn(Hkv, L, 128, generator=g).bfloat16()
    v = torch.randn(Hkv, L, 128, generator=g).bfloat16()
    return q, k, v


def _check(out, want):
    err = (out.float().cpu() - want.float()).abs()
    assert torch.isfinite(out.float()).all()
    assert err.max().item() <= OUT_MAX_ABS, err.max().item()
    assert err.mean().item() <= OUT_MEAN_ABS, err.mean().item()


@pytest.mark.parametrize(
    "shape",
    [(32, 8, 4096), (32, 8, 1), (32, 8, 31), (32, 8, 33), (8, 8, 1000), (28, 4, 5555), (32, 1, 700),
     (4, 2, 40000), (32, 8, 131072 + 17)],
)
def test_decode_matches_oracle(shape):
    from xattn.src.decode import single_decode_with_kv_cache

    H, Hkv, L = shape
    q, k, v = _mk(H, Hkv, L, 5, spread=3.0)
    out = single_decode_with_kv_cache(q.cuda(), k.cuda(), v.cuda(), kv_layout="HND")
    assert out.shape == (H, 128) and out.dtype == torch.bfloat16
    _check(out, O.single_decode_with_kv_cache(q, k, v, kv_layout="HND"))


def test_decode_layouts_views_and_scale():
    from xattn.src.decode import single_decode_with_kv_cache

    H, Hkv, L = 32, 8, 3000
    q, k, v = _mk(H, Hkv, L, 6)
    want = O.single_decode_with_kv_cache(q, k, v, kv_layout="HND", sm_scale=0.05)
    kc, vc = k.cuda(), v.cuda()
    # token-major cache
    out = single_decode_with_kv_cache(
        q.cuda(), kc.transpose(0, 1).contiguous(), vc.transpose(0, 1).contiguous(), kv_layout="NHD", sm_scale=0.05
    )
    _check(out, want)
    # a static cache longer than what is filled: sliced views, as the reference's forward passes them
    big_k = torch.zeros(Hkv, 4096, 128, dtype=torch.bfloat16, device="cuda")
    big_v = torch.full((Hkv, 4096, 128), float("nan"), dtype=torch.bfloat16, device="cuda")
    big_k[:, :L], big_v[:, :L] = kc, vc
    out = single_decode_with_kv_cache(q.cuda(), big_k[:, :L], big_v[:, :L], kv_layout="HND", sm_scale=0.05)
    _check(out, want)
    # caller-provided output and workspace
    from xattn.src import hip_backend as hb

    ws = torch.empty(hb.lib().xattn_decode_workspace_bytes(H, Hkv, L), dtype=torch.uint8, device="cuda")
    dst = torch.empty(H, 128, dtype=torch.bfloat16, device="cuda")
    got = single_decode_with_kv_cache(q.cuda(), kc, vc, kv_layout="HND", sm_scale=0.05, out=dst, workspace=ws)
    assert got is dst
    _check(dst, want)


def test_decode_is_last_row_of_prefill_kernel():
    from xattn.src.decode import single_decode_with_kv_cache
    from xattn.src.Xattention import block_sparse_attention

    g = torch.Generator().manual_seed(7)
    H, Hkv, L = 32, 8, 2048
    q = torch.randn(1, H, L, 128, generator=g).bfloat16().cuda()
    k = torch.randn(1, Hkv, L, 128, generator=g).bfloat16().cuda()
    v = torch.randn(1, Hkv, L, 128, generator=g).bfloat16().cuda()
    full = block_sparse_attention(q, k, v, causal=True)
    out = single_decode_with_kv_cache(q[0, :, -1], k[0], v[0], kv_layout="HND")
    assert (out.float() - full[0, :, -1].float()).abs().max().item() <= 1e-2


def test_decode_rejects_bad_arguments():
    from xattn.src import hip_backend as hb
    from xattn.src.decode import single_decode_with_kv_cache

    q, k, v = (t.cuda() for t in _mk(32, 8, 64, 8))
    with pytest.raises(ValueError):
        single_decode_with_kv_cache(q[:30], k, v, kv_layout="HND")          # 30 heads over 8
    with pytest.raises(KeyError):
        single_decode_with_kv_cache(q, k, v, kv_layout="DNH")
    with pytest.raises(hb.XattnHipError):
        single_decode_with_kv_cache(q.cpu(), k.cpu(), v.cpu(), kv_layout="HND")
    lib = hb.lib()
    assert lib.xattn_decode_workspace_bytes(32, 5, 64) == 0
    ws = torch.empty(16, dtype=torch.uint8, device="cuda")
    out = torch.empty(32, 128, dtype=torch.bfloat16, device="cuda")
    code = lib.xattn_decode_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), ws.data_ptr(), 16,
                                32, 8, 64, 128, 128, 64 * 128, 128, 64 * 128, 128, 128, 0.1, None)
    assert code == -7   # XATTN_ERR_WORKSPACE


# the last cache loaded with the default policy and the first of those loaded "not temporal" (more than 96 MiB), whose last tile
# has one key
@pytest.mark.parametrize("shape", [(32, 8, 24576), (32, 8, 24577), (28, 4, 49153)])
def test_decode_at_the_line_between_cache_policies(shape):
    from xattn.src.decode import single_decode_with_kv_cache

    H, Hkv, L = shape
    q, k, v = _mk(H, Hkv, L, L, spread=3.0)
    _check(single_decode_with_kv_cache(q.cuda(), k.cuda(), v.cuda(), kv_layout="HND"), O.single_decode_with_kv_cache(q, k, v, kv_layout="HND"))


# caches of one launch (up to 40 tiles of 32 keys, a wavefront every twelfth of them) and longer ones: tiles that lack keys, fewer
# tiles than parts and wavefronts, the edges of a wavefront's turns, groups of query heads that fill no copy of four rows, 32 and one;
# views whose heads and tokens lie apart
@pytest.mark.parametrize("H,Hkv,L", [
    (32, 8, 2), (32, 1, 5), (62, 2, 70), (3, 3, 32), (5, 1, 65), (32, 8, 96), (28, 4, 100), (32, 32, 129), (32, 1, 383), (64, 2, 384), (32, 8, 385), (14, 2, 416),
    (27, 9, 769), (32, 8, 1100), (40, 40, 1505), (32, 8, 1536), (32, 8, 1537), (28, 4, 1569), (130, 130, 1600), (257, 257, 40), (300, 300, 1700),
    # either side of the line, where every workgroup has a CU and where some wait
    (32, 8, 1280), (32, 8, 1281), (64, 64, 1280), (64, 64, 1281), (65, 65, 128), (65, 65, 129), (128, 128, 500), (257, 257, 129),
])
def test_decode_of_short_caches(H, Hkv, L):
    from xattn.src.decode import single_decode_with_kv_cache

    q, k, v = _mk(H, Hkv, L, L + H, spread=3.0)
    want = O.single_decode_with_kv_cache(q, k, v, kv_layout="HND")
    out = single_decode_with_kv_cache(q.cuda(), k.cuda(), v.cuda(), kv_layout="HND")
    _check(out, want)
    rows = torch.full((2 * H, 136), float("nan"), dtype=torch.bfloat16, device="cuda")
    rows[::2, :128] = q.cuda()
    cache = torch.full((2, L + 9, Hkv + 1, 144), float("nan"), dtype=torch.bfloat16, device="cuda")
    cache[0, :L, :Hkv, :128] = k.cuda().transpose(0, 1)
    cache[1, :L, :Hkv, :128] = v.cuda().transpose(0, 1)
    views = single_decode_with_kv_cache(rows[::2, :128], cache[0, :L, :Hkv, :128], cache[1, :L, :Hkv, :128], kv_layout="NHD")
    assert torch.equal(views, out)


# the decode step of an attention layer: caches [heads][tokens] and [tokens][heads], cut from larger ones, both kernels, and what
# has to go through the views instead
@pytest.mark.parametrize("H,Hkv,L", [(32, 8, 5), (32, 8, 1536), (32, 8, 1537), (4, 4, 9000), (28, 4, 33)])
def test_decode_of_a_layer(H, Hkv, L):
    from xattn.src import hip_backend as hb
    from xattn.src.decode import single_decode_with_kv_cache

    q, k, v = (t.cuda() for t in _mk(H, Hkv, L, L))
    want = single_decode_with_kv_cache(q, k, v, kv_layout="HND").reshape(1, 1, H * 128)
    step = q.reshape(1, 1, H, 128).transpose(1, 2)
    heads_first = torch.zeros(2, 1, Hkv, L + 50, 128, dtype=torch.bfloat16, device="cuda")
    heads_first[0, 0, :, :L], heads_first[1, 0, :, :L] = k, v
    tokens_first = heads_first.transpose(2, 3).contiguous().transpose(2, 3)
    for cache in (heads_first, tokens_first):
        got = hb.host().decode_layer(step, cache[0, :, :, :L], cache[1, :, :, :L])
        assert got.shape == (1, 1, H * 128) and torch.equal(got, want)
    ks, vs = heads_first[0, :, :, :L], heads_first[1, :, :, :L]
    for other in [(step.cpu(), ks, vs), (step.float(), ks, vs), (step, ks, vs[:, :, 1:]), (step, ks.transpose(2, 3), vs.transpose(2, 3)),
                  (step.expand(2, -1, -1, -1), ks, vs), (step.expand(-1, -1, 2, -1), ks, vs), (step[..., :64], ks, vs), (step[0], ks[0], vs[0])]:
        assert hb.host().decode_layer(*other) is None


# A short cache's probabilities are rounded to bf16 relative to the largest of their own 32 keys, which is then exact, whichever
# wavefront has the keys and in whatever order (relative to a running maximum the error against 64 bits is up to 4 % larger).  The
# same in 64 bits but for that rounding and the result's: what the kernel's 32-bit scores, of relative error 2^-22 or so, turn over of the
# roundings to 8 bits is one in some 10^4 of them by 2^-8 each, 10^-4 of the result
@pytest.mark.parametrize("H,Hkv,L", [(32, 8, 100), (32, 8, 400), (28, 4, 510), (32, 32, 640), (8, 1, 600)])
def test_short_caches_round_relative_to_a_tile(H, Hkv, L):
    from xattn.src.decode import single_decode_with_kv_cache

    q, k, v = _mk(H, Hkv, L, L)
    out = single_decode_with_kv_cache(q.cuda(), k.cuda(), v.cuda(), kv_layout="HND").cpu()
    g, tiles = H // Hkv, -(-L // 32)
    s = torch.full((Hkv, g, tiles * 32), -float("inf"), dtype=torch.float64)
    s[..., :L] = q.double().view(Hkv, g, 128) @ k.double().transpose(1, 2) / (128 ** 0.5 * 0.6931471805599453)
    s = s.view(Hkv, g, tiles, 32)
    own = s.amax(-1, keepdim=True)
    e, w = torch.exp2(s - own), torch.exp2(own - own.amax(2, keepdim=True))
    p = (e.bfloat16().double() * w).view(Hkv, g, -1)[..., :L]
    want = (p @ v.double() / (e * w).sum((2, 3))[..., None]).view(H, 128).bfloat16()
    assert ((out.double() - want.double()).norm() / want.double().norm()).item() <= 5e-4
