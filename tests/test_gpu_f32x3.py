"""float32 products on the bf16 matrix cores (three bf16 values an operand): projections and the codec's thin convs at the
edges of their tiles and of the rules that choose them, against 64-bit products.

Bound, per output, with S = sum_k |x_k w_k|: every accumulator addition rounds by at most 2^-24 of a partial sum (<= S),
6 per 32 products, the products left out are below 2^-25 S, and an input that went through ELU is off by an ulp."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _bound(s, K, extra=4):
    return (6 * K / 32 + extra) * 2.0 ** -24 * s + 1e-37


def _g(seed):
    return torch.Generator().manual_seed(seed)


@pytest.mark.parametrize("M,N,K", [(64, 10240, 64), (65, 5120, 32), (2500, 257, 96), (10304, 64, 64), (3000, 330, 160),
                                   (33, 10300, 64), (14080, 128, 32), (28200, 100, 32), (127, 5120, 512),
                                   (33, 16330, 32), (64, 16384, 64), (65, 8190, 96), (2500, 387, 96), (16321, 64, 64),
                                   (64, 16320, 64)])  # 256 workgroups of 64 x 64, and 255
@pytest.mark.parametrize("gelu", [False, True])
def test_linear_f32x3(gpu, M, N, K, gelu):
    from m3x import ops
    g = _g(M + N + K)
    x = torch.randn(M, K, generator=g).to(gpu)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(gpu)
    pw = ops.pack_weight(w)
    y = torch.full((M, N + 4), 7.0, device=gpu)[:, :N] if N % 4 == 0 else torch.full((M, N), 7.0, device=gpu)
    if gelu:
        ops.linear_act(x, pw, None, ops.ACT_GELU, y)
    else:
        ops.linear(x, pw, y)
    ref = x.double() @ w.double().t()
    bound = _bound(x.double().abs() @ w.double().abs().t(), K)
    if gelu:  # |gelu'| < 1.13; erf and its products a few ulp
        ref = F.gelu(ref)
        bound = 1.13 * bound + 2.0 ** -21 * ref.abs() + 2.0 ** -22
    assert bool(((y.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("M", [1, 2, 15, 16, 17])
@pytest.mark.parametrize("N,K", [(512, 512), (100, 32), (1537, 96), (512, 2048), (64, 4096), (48, 3584), (16400, 64),
                                 (33, 4128)])
@pytest.mark.parametrize("gelu", [False, True])
def test_linear_f32_few_rows(gpu, M, N, K, gelu):
    """Up to 16 rows: one workgroup of 16 K slices per tile (K up to 4096, up to 1024 tiles)."""
    from m3x import ops
    g = _g(M + N + K)
    x = torch.randn(M, K, generator=g).to(gpu)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(gpu)
    y = torch.full((M + 1, N), 7.0, device=gpu)
    pw = ops.pack_weight(w)
    ops.linear_act(x, pw, None, ops.ACT_GELU, y[:M]) if gelu else ops.linear(x, pw, y[:M])
    ref = x.double() @ w.double().t()
    bound = (K / 4 + 20) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())  # K / 4 additions and the slices'
    if gelu:
        ref = F.gelu(ref)
        bound = 1.13 * bound + 2.0 ** -21 * ref.abs() + 2.0 ** -22
    assert bool(((y[:M].double() - ref).abs() <= bound).all()) and bool((y[M] == 7.0).all())


def test_linear_f32x3_nonfinite(gpu):
    """Rows with infinities, NaN or values that bf16 rounds to infinity get what fp32 products give; the others are as
    without them."""
    from m3x import ops
    M, N, K = 700, 1024, 64
    g = _g(5)
    x = torch.randn(M, K, generator=g)
    x[3, 5], x[70, 0], x[131, 63], x[200, 7] = float("inf"), float("-inf"), float("nan"), 3.4e38
    w = (torch.randn(N, K, generator=g) * 0.1).abs() + 0.01
    x, w = x.to(gpu), w.to(gpu)
    y = ops.linear(x, ops.pack_weight(w))
    ref = x.double() @ w.double().t()
    assert bool((y[3] == float("inf")).all()) and bool((y[70] == float("-inf")).all()) and bool(y[131].isnan().all())
    assert torch.allclose(y[200].double(), ref[200], rtol=1e-6)
    rows = [r for r in range(M) if r not in (3, 70, 131, 200)]
    bound = _bound(x[rows].double().abs() @ w.double().abs().t(), K)
    assert bool(((y[rows].double() - ref[rows]).abs() <= bound).all())


@pytest.mark.parametrize("B,T,C,N,dil,pre", [(160, 96, 64, 64, 1, True), (80, 200, 32, 32, 1, True),
                                             (40, 480, 128, 64, 1, True), (100, 128, 32, 128, 8, False),
                                             (161, 97, 64, 32, 3, True), (20, 1000, 32, 64, 1, False),
                                             (90, 130, 32, 64, 1, True),  # half-empty row blocks: the fp32 kernel
                                             (7, 96, 64, 64, 1, True), (1, 1920, 64, 32, 1, True)])  # few workgroups
def test_conv_gemm_f32_gathered(gpu, B, T, C, N, dil, pre):
    from m3x import ops
    g = _g(B + T + C + N)
    k, pad = 3, 2 * dil
    x = torch.randn(B * T, C, generator=g).to(gpu)
    state = torch.randn(B + 2, pad * C + 8, generator=g).to(gpu)
    slots = torch.randperm(B + 2, generator=g)[:B].to(gpu)
    w = (torch.randn(N, k * C, generator=g) * (k * C) ** -0.5).to(gpu)
    bias, res = torch.randn(N, generator=g).to(gpu), torch.randn(B * T, N, generator=g).to(gpu)
    y = res.clone()
    ops.conv_gemm(x, ops.pack_weight(w), y, bias=bias, res=y, use_elu=True, gather=(state[:, :pad * C], slots, T, C, dil, pre))
    xd = x.double().view(B, T, C)
    j = torch.cat([state[slots, :pad * C].double().view(B, pad, C), F.elu(xd) if pre else xd], 1)
    cols = torch.cat([j[:, i * dil:i * dil + T] for i in range(k)], 2).view(B * T, k * C)
    pre_act = cols @ w.double().t() + bias.double() + res.double()
    bound = _bound(cols.abs() @ w.double().abs().t() + bias.double().abs() + res.double().abs(), k * C, 10) + 2.0 ** -22
    assert bool(((y.double() - F.elu(pre_act)).abs() <= bound).all())


@pytest.mark.parametrize("M,N,K", [(10240, 64, 32), (10303, 64, 96), (5130, 128, 64), (16000, 128, 32), (16321, 64, 96),
                                   (16320, 64, 96), (16321, 128, 64), (16320, 128, 64)])
def test_conv_gemm_f32_plain(gpu, M, N, K):
    from m3x import ops
    g = _g(M + N + K)
    x = torch.randn(M, K, generator=g).to(gpu)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(gpu)
    bias, y = torch.randn(N, generator=g).to(gpu), torch.randn(M, N, generator=g).to(gpu)
    ref = x.double() @ w.double().t() + bias.double() + y.double()
    bound = _bound(x.double().abs() @ w.double().abs().t() + bias.double().abs() + y.double().abs(), K, 10) + 2.0 ** -22
    ops.conv_gemm(x, ops.pack_weight(w), y, bias=bias, res=y, use_elu=True)
    assert bool(((y.double() - F.elu(ref)).abs() <= bound).all())


def _conv_case(B, seed):
    T, C, N = 96, 64, 64
    g = _g(seed)
    return (T, C, N, torch.randn(B * T, C, generator=g), torch.randn(B, 2 * C, generator=g),
            torch.randn(N, 3 * C, generator=g) * (3 * C) ** -0.5)


def test_nonfinite_rows_leave_the_others_alone(gpu):
    """A row with infinities, NaN or values that bf16 rounds to infinity (a stream that broke) does not change a bit of the
    other rows' (the other streams') results, in the projections, the plain conv and the gathered one."""
    from m3x import ops
    bad = torch.tensor([3, 70, 131, 200, 201, 699])
    g = _g(6)
    M, N, K = 700, 2048, 96
    x = torch.randn(M, K, generator=g)
    y = x.clone()
    y[bad, 5] = torch.tensor([float("inf"), float("-inf"), float("nan"), 3.4e38, -3.4e38, float("nan")])
    pw = ops.pack_weight(torch.randn(N, K, generator=g).to(gpu))
    rows = torch.ones(M, dtype=torch.bool)
    rows[bad] = False
    a, b = ops.linear(x.to(gpu), pw), ops.linear(y.to(gpu), pw)
    assert torch.equal(a[rows], b[rows])
    assert bool(b[3].isinf().all()) and bool(b[70].isinf().all()) and bool(b[131].isnan().all()) and bool(b[699].isnan().all())
    M = 16390
    x = torch.randn(M, 64, generator=g)
    y = x.clone()
    y[bad + 9000, 1] = float("nan")
    rows = torch.ones(M, dtype=torch.bool)
    rows[bad + 9000] = False
    pw = ops.pack_weight(torch.randn(64, 64, generator=g).to(gpu))
    a, b = (ops.conv_gemm(t.to(gpu), pw, torch.empty(M, 64, device=gpu)) for t in (x, y))
    assert torch.equal(a[rows], b[rows])
    B = 160
    T, C, N, x, state, w = _conv_case(B, 7)
    y, state_y = x.clone().view(B, T, C), state.clone()
    y[5, 40], y[17, 0], state_y[23] = float("nan"), float("inf"), float("nan")
    pw, slots = ops.pack_weight(w.to(gpu)), torch.arange(B, device=gpu)
    a, b = (ops.conv_gemm(t.reshape(B * T, C).to(gpu), pw, torch.empty(B * T, N, device=gpu),
                          gather=(s.to(gpu), slots, T, C, 1, True)).view(B, T, N) for t, s in ((x, state), (y, state_y)))
    clean = torch.ones(B, T, dtype=torch.bool)
    clean[5, 40:43] = clean[17, :3] = clean[23, :2] = False  # a row's three taps
    assert torch.equal(a[clean], b[clean]) and not bool(b[~clean].isfinite().all(1).any())


@pytest.mark.parametrize("e", [-60, -100, -112, -120, -126])
@pytest.mark.parametrize("which", ["x", "w"])
def test_tiny_operands(gpu, which, e):
    """Operands whose third (below 2^-110) or second bf16 value would be lost keep float32's accuracy: K / 4 additions and as
    many steps of the smallest number, which is 2^-149."""
    from m3x import ops
    M, N, K = 1030, 1024, 64
    g = _g(8)
    x, w = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g)
    T, C, CN, cx, state, cw = _conv_case(160, 9)
    if which == "x":
        x, cx, state = (t * 2.0 ** e for t in (x, cx, state))
    else:
        w, cw = w * 2.0 ** e, cw * 2.0 ** e
    def bound(s, k):
        return (k / 4 + 4) * (2.0 ** -24 * s + 2.0 ** -149)
    y = ops.linear(x.to(gpu), ops.pack_weight(w.to(gpu))).cpu().double()
    ref, s = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    assert bool(((y - ref).abs() <= bound(s, K)).all())
    slots = torch.arange(160, device=gpu)
    y = ops.conv_gemm(cx.to(gpu), ops.pack_weight(cw.to(gpu)), torch.empty(160 * T, CN, device=gpu),
                      gather=(state.to(gpu), slots, T, C, 1, False)).cpu().double()
    j = torch.cat([state.double().view(160, 2, C), cx.double().view(160, T, C)], 1)
    cols = torch.cat([j[:, i:i + T] for i in range(3)], 2).view(160 * T, 3 * C)
    ref, s = cols @ cw.double().t(), cols.abs() @ cw.double().abs().t()
    assert bool(((y - ref).abs() <= bound(s, 3 * C)).all())


def test_zero_rows_and_odd_columns(gpu):
    """Rows of zeros give zeros (signs and all finite), beside others, at a column count that is no multiple of 16."""
    from m3x import ops
    M, N, K = 2500, 515, 96
    g = _g(10)
    x, w = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g)
    x[100:300] = 0
    y = ops.linear(x.to(gpu), ops.pack_weight(w.to(gpu))).cpu().double()
    ref, s = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    assert not bool(y[100:300].any()) and bool(((y - ref).abs() <= _bound(s, K)).all())
