"""The work a serving engine has this framework do, as timed cases over the public surfaces.

A streaming engine drives, per 80 ms tick: one backbone step for its seats (sometimes with prompts prefilled in the
same step), the codebook-0 head and sampler, the depth transformer over codebooks 1..31, and the Mimi codec. The
families below are those calls, from one seat (latency) to a full GPU of 224 seats:

  step     StaticBackbone.step: one token for `seats` seats at ragged contexts (`ctx` their mean; `spread`: uniform
           in [64, 2 ctx], else Poisson). One seat runs the whole 28-layer model, as the latency of a lone stream
           is; more seats run a stack of 8 decoder layers.
  mixed    StaticBackbone.step_mixed: `seats` decoding seats and `prompts` prompts of `tokens` tokens in one step.
  prefill  StaticBackbone.prefill: a prompt of `tokens` tokens onto an empty slot, one step.
  cb0      codebook-0 head and sampler (Cb0Sampler.run) in a captured graph, as the frame step runs them.
  depth    FastDepth.run, the 31-codebook frame, in a captured graph, as the frame step runs it, with the logits of
           every level. `trunk` "swiglu" is the shared 4-layer SwiGLU / RMSNorm trunk in bf16; "depthv2" the
           11-group LayerNorm / GELU trunk with speaker constants in fp16, the engine's default.
  mimi     StaticMimi.decode: one frame for `seats` streams, `age` frames old (the attention window is full after
           125), in float32 (the codec's own precision) or float16.

Every pass starts from the same state: where a call advances a stream (a seat's length, a codec's tails and token
counts), run() puts those few words back first with plain copies, so a pass can be repeated.
"""
import functools
import math
import os
import random
import sys
from types import SimpleNamespace

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "maya2-native_amd"))
from m3x import ops, synth  # noqa: E402
from m3x.cb0 import Cb0Sampler  # noqa: E402
from m3x.serve.fast_backbone import StaticBackbone  # noqa: E402
from m3x.serve.fast_codec import StaticMimi  # noqa: E402
from m3x.serve.fast_depth import FastDepth  # noqa: E402
from m3x.staging import capture  # noqa: E402

DEV = "cuda"
# row buckets of a serving process: a batch is padded to the next one
BUCKETS = (1, 2, 4, 8, 16, 24, 32, 48, 64, 80, 96, 128, 160, 192, 224)
H, KV, D, HID, INTER, V = 16, 8, 128, 1024, 3072, 2048  # Qwen3-0.6B-shaped backbone; codebooks of 2048
LEVELS = 32
EPS = 1e-6


def listed():
    return [
        # a lone stream's backbone latency: the whole model, one row, a long context
        dict(name="step_1", family="step", seats=1, layers=28, ctx=2048, spread=False),
        # a part-filled GPU with streams of all ages
        dict(name="step_64_spread", family="step", seats=64, layers=8, ctx=1056, spread=True),
        # a full GPU in steady state
        dict(name="step_224", family="step", seats=224, layers=8, ctx=2048, spread=False),
        # a full GPU with new requests prefilled inline, 256 prompt tokens each: 2264 rows
        dict(name="mixed_216_8x256", family="mixed", seats=216, prompts=8, tokens=256, layers=8),
        # a new request's prompt, time to first audio
        dict(name="prefill_512", family="prefill", tokens=512, layers=8),
        # the head and sampler between backbone and depth at a full GPU; the smallest call
        dict(name="cb0_224", family="cb0", seats=224),
        # a lone stream's depth frame
        dict(name="depth_1", family="depth", seats=1, trunk="swiglu"),
        # a few streams on the engine's default depth
        dict(name="depth_16_v2", family="depth", seats=16, trunk="depthv2"),
        # a full GPU's depth frame
        dict(name="depth_224", family="depth", seats=224, trunk="swiglu"),
        # the codec for a lone stream, for a part-filled GPU in its faster precision, and for a full GPU
        dict(name="mimi_1", family="mimi", seats=1, age=130, dtype="float32"),
        dict(name="mimi_64_f16", family="mimi", seats=64, age=130, dtype="float16"),
        dict(name="mimi_224", family="mimi", seats=224, age=130, dtype="float32"),
    ]


def _logint(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    family = rng.choice(("step", "step", "mixed", "prefill", "cb0", "depth", "depth", "mimi", "mimi"))
    if family == "step":
        seats = _logint(rng, 1, 224)
        return dict(family=family, seats=seats, layers=28 if seats == 1 else 8, ctx=_logint(rng, 64, 2048),
                    spread=rng.random() < 0.5)
    if family == "mixed":
        return dict(family=family, seats=_logint(rng, 1, 216), prompts=rng.randint(1, 8),
                    tokens=_logint(rng, 16, 256), layers=8)
    if family == "prefill":
        return dict(family=family, tokens=_logint(rng, 16, 1024), layers=8)
    if family == "cb0":
        return dict(family=family, seats=_logint(rng, 1, 224))
    if family == "depth":
        trunk = rng.choice(("swiglu", "depthv2"))  # the 11-group trunk recomputes whole prefixes: fewer seats a GPU
        return dict(family=family, seats=_logint(rng, 1, 224 if trunk == "swiglu" else 80), trunk=trunk)
    return dict(family=family, seats=_logint(rng, 1, 224), age=rng.randint(2, 140),
                dtype=rng.choice(("float32", "float16")))


@torch.inference_mode()
def prepare(case, seed):
    return _PREPARE[case["family"]](case, seed)


@torch.inference_mode()  # a serving loop runs in it
def run(state):
    return state.run()


def _gen(seed, n=0):
    return torch.Generator(device=DEV).manual_seed(seed * 1009 + n)


def _normal(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device=DEV, dtype=dtype)


def _bucket(n):
    return next(b for b in BUCKETS if b >= n)


# ---------------------------------------------------------------- backbone
def _backbone(case, seed):
    return synth.qwen3_backbone(layers=case["layers"], seed=seed, device=DEV, gen=DEV, affine=synth.AFFINE)


def _contexts(case, seed):
    """(cached positions of each decoding seat, cached positions of each prompt's slot)."""
    rng = random.Random(seed)
    if case["family"] == "prefill":
        return [], [0]
    if case["family"] == "mixed":  # decoding seats of all ages; prompts follow a short voice prefix
        return ([min(4095, int(math.exp(rng.uniform(math.log(128), math.log(4096))))) for _ in range(case["seats"])],
                [rng.randint(0, 64) for _ in range(case["prompts"])])
    if case["seats"] == 1:
        return [case["ctx"] - 1], []
    if case["spread"]:
        lo = min(64, case["ctx"])
        return [rng.randint(lo, 2 * case["ctx"] - lo) for _ in range(case["seats"])], []
    return [max(1, int(round(rng.gauss(case["ctx"], math.sqrt(case["ctx"]))))) for _ in range(case["seats"])], []


def _cached(layer, seed, slots, capacity):
    """A layer's cached keys and values, N(0, 1)."""
    g = _gen(seed, 100 + layer)
    return tuple(_normal(g, slots, KV, capacity, D, dtype=torch.bfloat16) for _ in range(2))


def _step_inputs(case, seed):
    dec, pre = _contexts(case, seed)
    tokens = case.get("tokens", 0)
    capacity = max([c + 1 for c in dec] + [c + tokens for c in pre])
    g = _gen(seed, 1)
    x = _normal(g, len(dec), HID).to(torch.bfloat16)
    prompts = [_normal(g, tokens, HID).to(torch.bfloat16) for _ in pre]
    return dec, pre, -(-capacity // 128) * 128, x, prompts


def _prepare_step(case, seed):
    dec, pre, capacity, x, prompts = _step_inputs(case, seed)
    nd, n = len(dec), len(dec) + len(pre)
    rows = nd + sum(t.shape[0] for t in prompts)
    buckets = BUCKETS if not pre else (rows,)
    sb = StaticBackbone(_backbone(case, seed), n, capacity=capacity, batch_buckets=buckets, ctx_buckets=(capacity,),
                        attention="triton", fuse_proj=True, fuse_rope=True, fused_norm=True)
    for i in range(case["layers"]):
        k, v = _cached(i, seed, n, capacity)
        sb.k[i][:n].copy_(k)
        sb.v[i][:n].copy_(v)
    slots = list(range(nd))
    lengths = torch.tensor(dec + pre + [0], dtype=torch.long, device=DEV)
    host = dec + pre + [0]
    jobs = [(nd + j, t) for j, t in enumerate(prompts)]

    def rewind():
        sb.lengths.copy_(lengths)
        sb.lengths_cpu[:] = host

    def rows_of(slot, start, count, layers):  # views of the positions a call has written
        return [(sb.k[i][slot, :, start:start + count], sb.v[i][slot, :, start:start + count]) for i in layers]

    def go():
        rewind()
        if case["family"] == "prefill":
            return dict(h=sb.prefill(0, prompts[0]), kv=rows_of(0, 0, case["tokens"], range(case["layers"])))
        if pre:
            h, ends = sb.step_mixed(slots, x, jobs)
            return dict(h=h, ends=ends,
                        kv=[rows_of(nd + j, pre[j], case["tokens"], (case["layers"] - 1,)) for j in range(len(pre))])
        h = sb.step(slots, x)
        return dict(h=h, kv=rows_of(0, dec[0], 1, range(case["layers"])) if nd == 1 else [])

    rewind()
    # a serving process captures its graphs before its first request
    if pre:
        go()
    else:
        sb.warmup(batch_buckets=(_bucket(nd),))
    torch.cuda.synchronize()
    return SimpleNamespace(run=go, keep=sb)


def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _rope(x, pos):
    """x [T, heads, D]; the model's cos / sin tables are in its own dtype."""
    inv = 1.0 / (1e6 ** (torch.arange(0, D, 2, dtype=torch.int64).float() / D)).to(DEV)
    a = pos.float()[:, None] * inv[None]
    a = torch.cat([a, a], -1)
    cos, sin = (t.to(torch.bfloat16).double()[:, None] for t in (a.cos(), a.sin()))
    return x * cos + torch.cat([-x[..., D // 2:], x[..., :D // 2]], -1) * sin


def _exact_step(case, seed):
    dec, pre, capacity, x, prompts = _step_inputs(case, seed)
    lm = _backbone(case, seed).lm.model
    nd, n, T = len(dec), len(dec) + len(pre), case.get("tokens", 0)
    h = torch.cat([x] + prompts).double()
    pos = torch.cat([torch.tensor(dec, dtype=torch.long)] + [torch.arange(c, c + T) for c in pre]).to(DEV)
    spans = [(i, i + 1) for i in range(nd)] + [(nd + j * T, nd + (j + 1) * T) for j in range(len(pre))]
    starts = dec + pre
    written = []
    for i, layer in enumerate(lm.layers):
        a, m = layer.self_attn, layer.mlp
        w = lambda mod: mod.weight.double()  # noqa: E731
        y = _rms(h, w(layer.input_layernorm), EPS)
        q = _rope(_rms((y @ w(a.q_proj).t()).view(-1, H, D), w(a.q_norm), EPS), pos)
        k = _rope(_rms((y @ w(a.k_proj).t()).view(-1, KV, D), w(a.k_norm), EPS), pos)
        v = (y @ w(a.v_proj).t()).view(-1, KV, D)
        kc, vc = _cached(i, seed, n, capacity)
        o = torch.empty_like(q)
        rows = []
        for s, (r0, r1) in enumerate(spans):
            c, t = starts[s], r1 - r0
            keys = torch.cat([kc[s, :, :c].double(), k[r0:r1].transpose(0, 1)], 1)  # [KV, c + t, D]
            vals = torch.cat([vc[s, :, :c].double(), v[r0:r1].transpose(0, 1)], 1)
            qs = q[r0:r1].view(t, KV, H // KV, D).permute(1, 2, 0, 3).reshape(KV, -1, D)  # [KV, G * t, D]
            sc = torch.matmul(qs, keys.transpose(1, 2).contiguous()) * D ** -0.5
            if t > 1:
                seen = torch.arange(c + t, device=DEV)[None] <= torch.arange(c, c + t, device=DEV)[:, None]
                sc = sc.view(KV, H // KV, t, c + t).masked_fill(~seen, -math.inf).view(KV, -1, c + t)
            ov = torch.matmul(sc.softmax(-1), vals).view(KV, H // KV, t, D)
            o[r0:r1] = ov.permute(2, 0, 1, 3).reshape(t, H, D)
            if s >= nd or n == 1:
                rows.append((keys[:, c:], vals[:, c:]))
        written.append(rows)
        h = h + o.reshape(-1, H * D) @ w(a.o_proj).t()
        y = _rms(h, w(layer.post_attention_layernorm), EPS)
        h = h + (F.silu(y @ w(m.gate_proj).t()) * (y @ w(m.up_proj).t())) @ w(m.down_proj).t()
    out = _rms(h, lm.norm.weight.double(), EPS)
    if case["family"] == "prefill":
        return dict(h=out[-1], kv=[r[0] for r in written])
    if pre:
        return dict(h=out[:nd], ends=[out[r1 - 1] for _, r1 in spans[nd:]], kv=[[r] for r in written[-1]])
    return dict(h=out, kv=[r[0] for r in written] if nd == 1 else [])


def _work_step(case):
    L, T = case["layers"], case.get("tokens", 0)
    dec, pre = _contexts(case, 0)
    rows = len(dec) + len(pre) * T
    weights = (H + 2 * KV) * D * HID + H * D * HID + 3 * HID * INTER
    cached = sum(dec) + sum(pre)
    pairs = sum(c + 1 for c in dec) + sum(T * c + T * (T + 1) // 2 for c in pre)
    return dict(bytes=L * (2 * weights + 4 * KV * D * (cached + rows)) + 4 * rows * HID,
                flops=L * (2 * rows * weights + 4 * H * D * pairs))


# ---------------------------------------------------------------- sampling (codebook 0 and the depth)
def _sample(logits, u, temp, top_k):
    """Inverse CDF over the top-k set, largest first and by index among equals."""
    val, idx = torch.sort(logits.double() / temp, dim=-1, descending=True, stable=True)
    w = (val[:, :top_k] - val[:, :1]).exp()
    c = w.cumsum(-1)
    at = (c <= u.double()[:, None] * c[:, -1:]).sum(-1).clamp(max=top_k - 1)
    return idx.gather(1, at[:, None])[:, 0]


def _cb0_inputs(case, seed):
    g = _gen(seed, 2)
    head = _normal(g, V, HID).mul(0.1).to(torch.bfloat16)  # logits of standard deviation about 3
    return head, _normal(g, case["seats"], HID).to(torch.bfloat16), torch.rand(case["seats"], generator=g, device=DEV)


def _prepare_cb0(case, seed):
    head, h, u = _cb0_inputs(case, seed)
    n = case["seats"]
    cb = Cb0Sampler(head, n, temp=0.9, top_k=50, rep=0.0)
    b = cb.make_buffers(_bucket(n))
    b.slots[:n].copy_(torch.arange(n, device=DEV))
    b.h[:n].copy_(h)
    b.u[:n, 0].copy_(u)
    graph = capture(lambda: cb.run(b, uniforms=False), torch.cuda.graph_pool_handle())

    def go():
        graph.replay()
        return dict(logits=b.logits[:n], cb0=b.cb0[:n], stop=b.stop[:n])

    torch.cuda.synchronize()
    return SimpleNamespace(run=go, keep=cb)


def _exact_cb0(case, seed):
    head, h, u = _cb0_inputs(case, seed)
    logits = h.double() @ head.double().t()
    return dict(logits=logits, cb0=_sample(logits, u, 0.9, 50), stop=None)


def _work_cb0(case):
    n = case["seats"]
    return dict(bytes=2 * (V * HID + n * HID + n * V) + 24 * n, flops=2 * n * V * HID)


# ---------------------------------------------------------------- depth
_DEPTH = dict(swiglu=dict(dtype=torch.bfloat16, temp=0.9, top_k=50, heads=8, ffn=2816),
              depthv2=dict(dtype=torch.float16, temp=0.7, top_k=64, heads=16, ffn=3072))
_PEAK = 0.02


@functools.lru_cache(maxsize=2)
def _depth_model(trunk):
    """A depth model that is as sure of its codes as a trained one: each level's head holds, beside its random rows, a
    multiple of the embedding of the code one step before, so one code stands well above the rest and a change of
    rounding does not change the codes that the later levels continue from."""
    if trunk == "swiglu":
        m = synth.swiglu_depth(seed=1, device=DEV, gen=DEV, affine=synth.AFFINE)
        d = m.depth
        d.embed.mul_(50)
        emb = d.embed.double()
    else:
        m = synth.depthv2_like(seed=2, device=DEV, dtype=torch.float16, affine_std=0.1)
        d = m.depth
        d.code_lo.weight.mul_(50)
        d.code_up.weight.mul_(128 ** -0.5 / 0.02)
        emb = (d.code_lo.weight.double() @ d.code_up.weight.double().t()).view(LEVELS - 1, V, HID)
    for lv, head in enumerate(d.heads):
        head.weight = (head.weight.double() + _PEAK * emb[lv].roll(7 * lv + 1, 0)).to(head.weight.dtype)
    return m


def _depth_inputs(case, seed):
    n, spec = case["seats"], _DEPTH[case["trunk"]]
    g = _gen(seed, 3)
    return SimpleNamespace(h=_normal(g, n, HID).to(spec["dtype"]),
                           cb0=torch.randint(0, V, (n,), generator=g, device=DEV),
                           u=torch.rand(n, LEVELS - 1, generator=g, device=DEV),
                           mem=_normal(g, n, HID).to(spec["dtype"]))


def _prepare_depth(case, seed):
    n, spec, x = case["seats"], _DEPTH[case["trunk"]], _depth_inputs(case, seed)
    fd = FastDepth(_depth_model(case["trunk"]), n, dtype=spec["dtype"], temp=spec["temp"], top_k=spec["top_k"],
                   batch_buckets=BUCKETS, fused=True)
    one = torch.ones(1, 1, device=DEV)
    for s in range(n):
        fd.set_speaker(s, x.mem[s].view(1, 1, HID), one)
    b = fd.make_buffers(fd.bucket_for(n))
    b.table.stage(dict(slot=range(n)))
    b.h[:n].copy_(x.h)
    b.codes[:n, 0].copy_(x.cb0)
    b.u[:n].copy_(x.u)
    logits = []

    def frame():
        logits.clear()
        fd.run(b, uniforms=False, trace=logits)

    graph = capture(frame, torch.cuda.graph_pool_handle())

    def go():
        graph.replay()
        return dict(codes=b.codes[:n], feedback=b.feedback[:n], logits=[t[:n] for t in logits])

    torch.cuda.synchronize()
    return SimpleNamespace(run=go, keep=fd)


def _exact_depth(case, seed):
    n, spec, x = case["seats"], _DEPTH[case["trunk"]], _depth_inputs(case, seed)
    m = _depth_model(case["trunk"])
    d, heads = m.depth, spec["heads"]
    hd = HID // heads
    w = lambda mod: mod.weight.double()  # noqa: E731

    def norm(t, mod):
        if mod.bias is None:
            return _rms(t, w(mod), mod.eps)
        return F.layer_norm(t, (HID,), w(mod), mod.bias.double(), mod.eps)

    if case["trunk"] == "swiglu":
        first, embed = d.level0.double(), lambda lv, code: d.embed[lv][code].double()
        cross = [0.0] * len(d.groups[0])
    else:
        lvl, up = w(d.level_emb), w(d.code_up).t()
        first = lvl[0]
        embed = lambda lv, code: w(d.code_lo)[code + lv * V] @ up + lvl[lv + 1]  # noqa: E731
        cross = [((x.mem.double() @ w(c.kv).t())[:, HID:] @ w(c.o).t())[:, None] for c in d.cross]
    prefix = torch.empty(n, LEVELS, HID, dtype=torch.float64, device=DEV)
    prefix[:, 0] = x.h.double() @ w(d.in_proj).t() + first
    codes, logits = [x.cb0], []
    for level in range(1, LEVELS):
        prefix[:, level] = embed(level - 1, codes[-1])
        t, T = prefix[:, :level + 1], level + 1
        mask = torch.ones(T, T, dtype=torch.bool, device=DEV).tril()
        for li, blk in enumerate(d.groups[d.group_of_level[level]]):
            q, k, v = ((norm(t, blk.n1) @ w(blk.qkv).t()).view(n, T, 3, heads, hd).permute(2, 0, 3, 1, 4))
            sc = torch.matmul(q, k.transpose(2, 3).contiguous()) * hd ** -0.5
            a = torch.matmul(sc.masked_fill(~mask, -math.inf).softmax(-1), v.contiguous())
            t = t + a.transpose(1, 2).reshape(n, T, HID) @ w(blk.o).t()
            y = norm(t, blk.n2)
            if case["trunk"] == "swiglu":
                gate, up_ = (y @ w(blk.gate_up).t()).chunk(2, -1)
                t = t + (F.silu(gate) * up_) @ w(blk.down).t()
            else:
                t = t + F.gelu(y @ w(blk.f1).t()) @ w(blk.f2).t()
            t = t + cross[li]
        logits.append(norm(t[:, -1], d.norm) @ w(d.heads[level - 1]).t())
        codes.append(_sample(logits[-1], x.u[:, level - 1], spec["temp"], spec["top_k"]))
    codes = torch.stack(codes, 1)
    table = m.audio_in.table.weight.double()
    fb = sum(table[codes[:, lv] + V * lv] for lv in range(LEVELS)) / math.sqrt(LEVELS)
    return dict(codes=codes, feedback=_rms(fb, w(m.audio_in.norm), m.audio_in.norm.eps), logits=logits)


def _work_depth(case):
    n, spec = case["seats"], _DEPTH[case["trunk"]]
    swiglu = case["trunk"] == "swiglu"
    layer = 4 * HID * HID + (3 if swiglu else 2) * HID * spec["ffn"]
    # positions evaluated: one a level, and a whole prefix where a level starts a weight group (levels 1-9, 17 and 25
    # of the 11-group trunk), the last layer at the last position only
    starts = (1,) if swiglu else tuple(range(1, 10)) + (17, 25)
    rows = (LEVELS - 1 - len(starts)) * 4 * n + sum(3 * (lv + 1) + 1 for lv in starts) * n
    groups = 1 if swiglu else 11
    head = (LEVELS - 1) * V * HID
    return dict(bytes=2 * (4 * groups * layer + head + n * LEVELS * (2 * HID + V)),
                flops=2 * rows * layer + 2 * n * head)


# ---------------------------------------------------------------- codec
@functools.lru_cache(maxsize=1)
def _mimi_model():
    return synth.mimi(seed=7, device=DEV)


def _mimi_codes(case, seed):
    return torch.randint(0, V, (case["seats"], 32, case["age"] + 1), generator=_gen(seed, 4), device=DEV)


def _prepare_mimi(case, seed):
    n, codes = case["seats"], _mimi_codes(case, seed)
    sm = StaticMimi(_mimi_model(), n, batch_buckets=BUCKETS, dtype=getattr(torch, case["dtype"]))
    slots = list(range(n))
    for t in range(case["age"]):
        sm.decode(slots, codes[:, :, t])
    last = codes[:, :, -1].contiguous()
    held = (sm.conv_flat, sm.key_pos, sm.tokens)
    saved = [t.clone() for t in held]

    def go():
        # the stream back at the frame's start; the rows a frame adds to the attention rings replace ones that lie
        # outside its window, so they are the same after each pass
        for t, s in zip(held, saved):
            t.copy_(s)
        return sm.decode(slots, last)

    torch.cuda.synchronize()
    return SimpleNamespace(run=go, keep=sm)


def _conv(x, mod):
    """Causal stride-one convolution of x [B, C, T] as one product in 64 bits."""
    c = mod.conv
    k, dil = c.kernel_size[0], c.dilation[0]
    j = F.pad(x, ((k - 1) * dil, 0))
    cols = torch.cat([j[:, :, i * dil:i * dil + x.shape[2]] for i in range(k)], 1)  # [B, k * C, T]
    w = c.weight.double().permute(0, 2, 1).reshape(c.out_channels, -1)
    y = torch.matmul(cols.transpose(1, 2).contiguous(), w.t()).transpose(1, 2)
    return y if c.bias is None else y + c.bias.double()[:, None]


def _conv_t(x, c):
    """Causal transposed convolution (the overflow past the last frame is cut)."""
    B, cin, T = x.shape
    k, s = c.kernel_size[0], c.stride[0]
    if c.groups > 1:
        cols = x[:, :, :, None] * c.weight.double()[:, 0][None, :, None]  # [B, C, T, k]
    else:
        w = c.weight.double().reshape(cin, -1)
        cols = torch.matmul(x.transpose(1, 2).contiguous(), w).view(B, T, c.out_channels, k).transpose(1, 2)
    y = x.new_zeros(B, cols.shape[1], T * s + k - s)
    for i in range(k):
        y[:, :, i:i + T * s:s] += cols[..., i]
    y = y[:, :, :T * s]
    return y if c.bias is None else y + c.bias.double()[:, None]


def _exact_mimi(case, seed):
    return torch.cat([_exact_mimi_seats(c) for c in _mimi_codes(case, seed).split(16)])


def _exact_mimi_seats(codes):
    m = _mimi_model()
    q = m.quantizer
    sem, ac = q.semantic_residual_vector_quantizer, q.acoustic_residual_vector_quantizer
    rows = lambda layers, at: sum(l.codebook.embed.double()[codes[:, at + i]] for i, l in enumerate(layers))  # noqa: E731
    x = (rows(sem.layers, 0) @ sem.output_proj.weight.double()[:, :, 0].t()
         + rows(ac.layers, 1) @ ac.output_proj.weight.double()[:, :, 0].t()).transpose(1, 2)
    x = _conv_t(x, m.upsample.conv).transpose(1, 2)  # [B, T, 512]
    B, T, C = x.shape
    rot, nh = m.decoder_transformer.rotary_emb, m.config.num_attention_heads
    pos = torch.arange(T, device=DEV)
    ang = (pos.float()[:, None] * rot.inv_freq.float().to(DEV)[None]).double()
    ang = torch.cat([ang, ang], -1)
    cos, sin = ang.cos() * rot.attention_scaling, ang.sin() * rot.attention_scaling
    seen = (pos[None] <= pos[:, None]) & (pos[None] > pos[:, None] - m.config.sliding_window)
    turn = lambda t: t * cos + torch.cat([-t[..., t.shape[-1] // 2:], t[..., :t.shape[-1] // 2]], -1) * sin  # noqa: E731
    norm = lambda t, n: F.layer_norm(t, (C,), n.weight.double(), n.bias.double(), n.eps)  # noqa: E731
    for L in m.decoder_transformer.layers:
        a, y = L.self_attn, norm(x, L.input_layernorm)
        qh, kh, vh = ((y @ p.weight.double().t()).view(B, T, nh, -1).transpose(1, 2)
                      for p in (a.q_proj, a.k_proj, a.v_proj))
        sc = torch.matmul(turn(qh), turn(kh).transpose(2, 3).contiguous()) * qh.shape[-1] ** -0.5
        o = torch.matmul(sc.masked_fill(~seen, -math.inf).softmax(-1), vh.contiguous())
        o = o.transpose(1, 2).reshape(B, T, C) @ a.o_proj.weight.double().t()
        x = x + L.self_attn_layer_scale.scale.double() * o
        y = F.gelu(norm(x, L.post_attention_layernorm) @ L.mlp.fc1.weight.double().t())
        x = x + L.mlp_layer_scale.scale.double() * (y @ L.mlp.fc2.weight.double().t())
    # the convolutions reach back less than 16 positions
    mods, back = list(m.decoder.layers), min(T, 18)
    x = x.transpose(1, 2)[:, :, T - back:]
    x = _conv(x, mods[0])
    i = 1
    while i < len(mods) - 2:
        x = _conv_t(F.elu(x), mods[i + 1].conv)
        blk = list(mods[i + 2].block)
        x = x + _conv(F.elu(_conv(F.elu(x), blk[1])), blk[3])
        i += 3
    return _conv(F.elu(x), mods[i + 1])[:, 0, -1920:]


def _work_mimi(case):
    n, e = case["seats"], 4 if case["dtype"] == "float32" else 2
    C, t = 512, 2  # transformer width, tokens a frame
    params = 2 * 256 * C + C * 4 + 8 * 12 * C * C
    macs = t * 8 * 12 * C * C + 2 * 256 * C
    ch = 1024  # SEANet: conv 7, then transposed convolutions by 8, 6, 5, 4, each with a residual block, then conv 3
    params += 7 * C * ch
    macs += t * 7 * C * ch
    for s in (8, 6, 5, 4):
        params += 2 * s * ch * ch // 2
        macs += t * 2 * s * ch * ch // 2
        ch, t = ch // 2, t * s
        params += 3 * ch * ch // 2 + ch // 2 * ch
        macs += t * (3 * ch * ch // 2 + ch // 2 * ch)
    keys = min(250, 2 * case["age"])
    rings = 8 * 2 * C * e * keys
    return dict(bytes=e * params + n * (rings + 32 * 256 * e + 32 * 8 + 4 * 1920),
                flops=2 * n * (macs + 8 * 2 * 2 * C * (keys + 2) + 1920 * 3 * 64))


# ---------------------------------------------------------------- tolerances
def tolerance(case):
    """About four times the distance measured between each path and its 64-bit evaluation (bf16 backbone: 0.0085 over
    8 layers, 0.017 over 28; bf16 depth logits 0.006; fp16 depth 0.0006, its bf16 feedback row 0.0029; head 0.0017;
    codec 1.4e-6 in float32, 0.0016 in float16). A code changes when a change of rounding moves a step of its
    distribution across its uniform: about one draw in 50 at the flat logits of the head, hardly any in the depth."""
    family = case["family"]
    if family == "mimi":
        return {"rel": 6e-6 if case["dtype"] == "float32" else 7e-3}
    if family == "cb0":
        return {"rel": 7e-3, "differ": 0.1}
    if family == "depth":
        return {"rel": 0.025 if case["trunk"] == "swiglu" else 0.012, "differ": 0.01}
    return {"rel": 0.07 if case["layers"] > 8 else 0.035}


@torch.inference_mode()
def exact(case, seed):
    return _EXACT[case["family"]](case, seed)


def work(case):
    return _WORK[case["family"]](case)


_PREPARE = dict(step=_prepare_step, mixed=_prepare_step, prefill=_prepare_step, cb0=_prepare_cb0, depth=_prepare_depth,
                mimi=_prepare_mimi)
_EXACT = dict(step=_exact_step, mixed=_exact_step, prefill=_exact_step, cb0=_exact_cb0, depth=_exact_depth,
              mimi=_exact_mimi)
_WORK = dict(step=_work_step, mixed=_work_step, prefill=_work_step, cb0=_work_cb0, depth=_work_depth, mimi=_work_mimi)
