"""The column-strip projections at the edges of the rule that chooses their tiles (257 rows, 512 / 513 rows, each tile, odd
rows and columns), against float64 products.

Bounds: one rounding to the storage type is at most e = 2^-8 (bf16, 8 significant bits) or 2^-11 (fp16, 11) of the value;
the fp32 sums add K 2^-24 of the summed magnitudes."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
SHAPES = [(257, 4096, 1024), (300, 1040, 64), (511, 3072, 1024), (512, 2816, 128), (513, 1000, 192), (640, 1024, 2048),
          (1030, 256, 1536), (1111, 3000, 64), (2264, 4096, 128), (7700, 500, 64), (4800, 3200, 64), (700, 2360, 64),
          (3136, 3072, 1024), (512, 1000, 2048), (300, 512, 2048), (352, 2048, 512), (384, 2048, 512)]


def _data(M, N, K, dtype, gpu, n=1):
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).to(dtype).to(gpu)
    ws = [(torch.randn(N, K, generator=g) * K ** -0.5).to(dtype).to(gpu) for _ in range(n)]
    return x, ws


def _prod(x, w):
    return x.double() @ w.double().t(), (x.double().abs() @ w.double().abs().t()) * x.shape[1] * 2.0 ** -24


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_strip_plain_and_gelu(gpu, M, N, K, dtype):
    from m3x import ops
    e = EPS[dtype]
    x, (w,) = _data(M, N, K, dtype, gpu)
    ref, acc = _prod(x, w)
    y = ops.linear(x, ops.pack_weight(w)).double()
    assert bool(((y - ref).abs() <= e * ref.abs() + acc + 1e-7).all())
    y = ops.linear_act(x, ops.pack_weight(w), None, ops.ACT_GELU).double()
    gref = F.gelu(ref)
    assert bool(((y - gref).abs() <= 1.13 * (e * ref.abs() + acc) + e * gref.abs() + 1e-6).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(260, 3072, 256), (400, 2816, 64), (512, 1536, 128), (513, 900, 64), (700, 3072, 64),
                                   (1500, 3072, 128), (3000, 1000, 64)])
def test_strip_swiglu(gpu, M, N, K, dtype):
    from m3x import ops
    e = EPS[dtype]
    x, (wg, wu) = _data(M, N, K, dtype, gpu, 2)
    (g, ag), (u, au) = _prod(x, wg), _prod(x, wu)
    y = ops.linear_act(x, ops.pack_weight(wg), ops.pack_weight(wu), ops.ACT_SWIGLU).double()
    s = F.silu(g)
    bound = (1.1 * (e * g.abs() + ag) + 1.01 * e * s.abs()) * u.abs() * 1.01 + s.abs() * (e * u.abs() + au) * 1.02
    assert bool(((y - s * u).abs() <= bound + 1.01 * e * (s * u).abs() + 1e-6).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(300, 1024, 2048), (512, 1024, 2048), (513, 1024, 1024), (1100, 1024, 3072),
                                   (2264, 1024, 2048), (999, 2048, 64), (512, 2048, 128)])
def test_strip_resid(gpu, M, N, K, dtype):
    from m3x import ops
    e = EPS[dtype]
    x, (w,) = _data(M, N, K, dtype, gpu)
    h = torch.randn(M, N, generator=torch.Generator().manual_seed(M)).to(dtype).to(gpu)
    out = torch.empty_like(h)
    part = torch.empty(ops.tile_stats_elems(M, N), device=gpu)
    ops.linear_resid(x, ops.pack_weight(w), h, out, part, ops.NORM_RMS)
    p, acc = _prod(x, w)
    ref = h.double() + p
    assert bool(((out.double() - ref).abs() <= (e * p.abs() + acc) * 1.01 + e * ref.abs() * 1.01 + 1e-6).all())
    t = out.double().view(M, N // 16, 16)
    st = part.view(M, N // 16, 2).double()
    assert torch.allclose(st[..., 0], t.sum(-1), atol=1e-4, rtol=0) and torch.allclose(st[..., 1], t.square().sum(-1), rtol=1e-5)


@pytest.mark.parametrize("M", [257, 320, 511, 640, 1030, 2264])
def test_strip_qk_rope_matches_two_launches(gpu, M):
    """The fused projection + q/k norm + RoPE + cache write gives the two launches' bits at every tile it takes."""
    from m3x import ops
    H, KV, D, K = 16, 8, 128, 1024
    x, (w,) = _data(M, (H + 2 * KV) * D, K, torch.bfloat16, gpu)
    pw = ops.pack_weight(w)
    g = torch.Generator().manual_seed(M)
    cos, sin = (torch.randn(M + 8, D, generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    wq, wk = (torch.randn(D, generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    slots = torch.randint(0, 3, (M,), generator=g).to(gpu)
    pos = torch.arange(M, dtype=torch.int32, device=gpu)
    outs = []
    for fused in (True, False):
        kc, vc = (torch.zeros(3, KV, M + 8, D, dtype=torch.bfloat16, device=gpu) for _ in range(2))
        q = torch.zeros(M, H, D, dtype=torch.bfloat16, device=gpu)
        qkv = torch.zeros(M, (H + 2 * KV) * D, dtype=torch.bfloat16, device=gpu)
        args = (qkv, q, kc, vc, slots, pos, cos, sin, wq, wk, 1e-6, H, KV)
        if fused:
            ops.linear_qk_rope(x, pw, *args)
            if M > 512:
                assert not qkv.any()  # the staging buffer is left alone
            else:
                assert torch.equal(qkv, ops.linear(x, pw))
        else:
            ops.linear(x, pw, qkv)
            ops.qk_norm_rope_cache(*args)
        outs.append((q, kc, vc))
    assert all(torch.equal(a, b) for a, b in zip(*outs))
