"""The codec's ring attention against float64: every wave of its workgroup with live entries, rings of 256 and of sizes that
are no multiple of 64, positions before, at and past the wrap, this call's rows across a wave's edge (63 / 64) and across the
ring's end, one and two tokens, and both sides of the size from which the rows are streamed (32 MB of keys and values).

Bound, with S = 0.125 sum |q| |k| of a key and e the storage type's rounding: RoPE rounds a query by 4 steps, a score's products
and sums by 12, so a score is off by at most 16 2^-24 max S and a probability by twice that and 4 steps; an output adds the 8
rows a lane holds, 3 lane steps and 4 waves, the sum of the probabilities as many, and the quotient is rounded once to the
storage type: (32 max S + 40) 2^-24 sum p |v| + e |out|."""
import pytest
import torch

pytestmark = pytest.mark.gpu
E = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}
H, HD = 8, 64
NEVER = -(1 << 40)
STARTS = (0, 1, 5, 31, 63, 64, 127, 128, 191, 200, 249, 250, 251, 252, 253, 255, 256, 315, 319, 400, 503, 504, 511, 1000, 1087)


def _state(gpu, dtype, B, T, ring, window, seed):
    """B seats on permuted slots, each with the ring that a stream of p0 tokens has: entry p % ring holds position p."""
    g = torch.Generator().manual_seed(seed)
    S = B + 2
    p0 = torch.tensor([STARTS[i % len(STARTS)] for i in range(B)])
    slots = torch.randperm(S, generator=g)[:B]
    kr, vr = (torch.randn(S, ring, H, HD, generator=g).to(dtype) for _ in range(2))
    tokens, kp = torch.zeros(S, dtype=torch.long), torch.full((S, ring), NEVER)
    j = torch.arange(ring)[None]
    last = p0[:, None] - 1 - (p0[:, None] - 1 - j) % ring
    tokens[slots], kp[slots] = p0, torch.where(last >= 0, last, NEVER)
    qkv = torch.randn(B * T, 3 * H * HD, generator=g).to(dtype)
    inv_freq = 10000.0 ** (-torch.arange(0, HD, 2) / HD)
    return SimpleState(gpu, dtype, B, T, ring, window, p0, slots, kr, vr, kp, tokens, qkv, inv_freq.float())


class SimpleState:
    def __init__(self, gpu, dtype, B, T, ring, window, p0, slots, *tensors):
        self.dtype, self.B, self.T, self.ring, self.window, self.p0 = dtype, B, T, ring, window, p0
        self.slots = slots.to(gpu)
        self.kr, self.vr, self.kp, self.tokens, self.qkv, self.inv_freq = (t.to(gpu) for t in tensors)

    def run(self):
        from m3x import ops
        out = torch.full((self.B * self.T, H * HD), 7.0, dtype=self.dtype, device=self.qkv.device)
        ops.ring_attn(self.qkv, self.kr, self.vr, self.kp, self.tokens, self.slots, self.inv_freq, 1.0, out, self.B, self.T,
                      H, self.ring, self.window)
        return out

    def positions(self):  # [B, T]
        return self.p0.to(self.slots.device)[:, None] + torch.arange(self.T, device=self.slots.device)


def _rope(x, pos, inv_freq):
    """x [B, T, H, 64] float64; the angle as the float32 product the codec defines."""
    ang = (pos.float()[..., None] * inv_freq).double()
    cos, sin = (torch.cat([f(ang)] * 2, -1)[:, :, None] for f in (torch.cos, torch.sin))
    return x * cos + torch.cat([-x[..., 32:], x[..., :32]], -1) * sin


@pytest.mark.parametrize("ring,window", [(256, 250), (252, 251), (100, 64), (8, 6)])
@pytest.mark.parametrize("T", [1, 2])
@pytest.mark.parametrize("dtype,B", [(torch.float32, 25), (torch.float32, 34), (torch.float16, 25), (torch.float16, 67),
                                     (torch.bfloat16, 25), (torch.bfloat16, 67)])
def test_ring_attn(gpu, dtype, B, T, ring, window):
    s = _state(gpu, dtype, B, T, ring, window, B + T + ring)
    k0, v0, kp0, tok0 = (t.clone() for t in (s.kr, s.vr, s.kp, s.tokens))
    out = s.run().double().view(B, T, H, HD)
    pos, at = s.positions(), s.positions() % ring
    x = s.qkv.double().view(B, T, 3, H, HD)
    # this call's rows: the rotated keys within their rounding, the values and positions as given, nothing else touched
    rows = s.slots[:, None].expand(B, T)
    knew = _rope(x[:, :, 1], pos, s.inv_freq)
    assert bool(((s.kr[rows, at].double() - knew).abs() <= E[dtype] * knew.abs() + 4 * 2.0 ** -24 * x[:, :, 1].abs().amax(-1, True)).all())
    k0[rows, at], v0[rows, at], kp0[rows, at] = s.kr[rows, at], x[:, :, 2].to(dtype), pos
    assert torch.equal(s.kr, k0) and torch.equal(s.vr, v0) and torch.equal(s.kp, kp0) and torch.equal(s.tokens, tok0)
    q = _rope(x[:, :, 0], pos, s.inv_freq)
    k, v = s.kr[s.slots].double(), s.vr[s.slots].double()  # [B, ring, H, 64]
    score = torch.einsum("bthd,bjhd->bthj", q, k) * 0.125
    mag = torch.einsum("bthd,bjhd->bthj", q.abs(), k.abs()) * 0.125
    kp = s.kp[s.slots][:, None, None, :]
    seen = (kp <= pos[:, :, None, None]) & (kp > pos[:, :, None, None] - window)
    p = score.masked_fill(~seen, float("-inf")).softmax(-1)
    ref = torch.einsum("bthj,bjhd->bthd", p, v)
    worst = mag.masked_fill(~seen, 0).amax(-1, True)
    bound = (32 * worst + 40) * 2.0 ** -24 * torch.einsum("bthj,bjhd->bthd", p, v.abs()) + E[dtype] * ref.abs() + 1e-7
    bad = (out - ref).abs() > bound
    assert not bool(bad.any()), [(int(b), STARTS[int(b) % len(STARTS)]) for b in bad.flatten(1).any(1).nonzero()]


@pytest.mark.parametrize("dtype,B", [(torch.float32, 25), (torch.float32, 34), (torch.float16, 25), (torch.float16, 67)])
@pytest.mark.parametrize("ring,window", [(256, 250), (100, 64), (8, 6)])
def test_rows_out_of_sight_have_no_effect(gpu, dtype, B, ring, window):
    """What lies in entries that a token does not see (an earlier stream's rows, rows that left the window, the next token's
    own) does not reach its output, infinities and NaN included."""
    a, b = (_state(gpu, dtype, B, 2, ring, window, 3) for _ in range(2))
    stale = (b.kp[b.slots] <= b.positions()[:, :1] - window) | (b.kp[b.slots] < 0)  # seen by neither token
    for t in (b.kr, b.vr):
        rows = t[b.slots]
        rows[stale] = float("nan")
        rows[:, 1::2][stale[:, 1::2]] = float("inf")
        t[b.slots] = rows
    ref, got = a.run(), b.run()
    assert torch.equal(ref, got)
    # the first token sees neither the second's value nor its key; the second does not see the row that left the window
    c = _state(gpu, dtype, B, 2, ring, window, 3)
    c.qkv.view(B, 2, 3, H * HD)[:, 1, 2] = float("nan")
    assert torch.equal(c.run().view(B, 2, -1)[:, 0], ref.view(B, 2, -1)[:, 0])
    d = _state(gpu, dtype, B, 2, ring, window, 3)
    leaving = d.kp[d.slots] == d.positions()[:, :1] - window + 1
    assert bool(leaving.any())
    rows = d.vr[d.slots]
    rows[leaving] = float("nan")
    d.vr[d.slots] = rows
    assert torch.equal(d.run().view(B, 2, -1)[:, 1], ref.view(B, 2, -1)[:, 1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_reset_slot_forgets_a_broken_stream(gpu, dtype):
    """A stream whose values overflowed leaves infinities and NaN in its ring; after reset() the slot's next stream is that of
    a fresh slot."""
    from m3x import synth
    from m3x.serve.fast_codec import StaticMimi
    sm = StaticMimi(synth.mimi(seed=35, device=gpu), 2, batch_buckets=(2,), use_graphs=False, dtype=dtype)
    codes = synth.mimi_codes(1, 3, seed=36).to(gpu)
    with torch.inference_mode():
        sm.kv[:, :, 0] = float("nan")
        sm.reset(0)
        for t in range(3):
            c = codes[:1, :, t].expand(2, -1)
            pcm = sm.decode([0, 1], c)
            assert bool(pcm.isfinite().all()) and torch.equal(pcm[0], pcm[1]), t
