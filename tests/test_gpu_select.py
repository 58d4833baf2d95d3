"""The samplers' candidate selection at the edges of its paths (the threads' maxima up to k = 128, the histogram above,
the radix select as the fallback of both), bit-exact against the C oracle: the kept set, its order and the draw are the
contract's whatever candidates a path lets through."""
import numpy as np
import pytest
import torch

from helpers import bf16_bits
from oracle import coracle as C

pytestmark = pytest.mark.gpu


def _rows(V, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(24, V, generator=g) * 2
    x[1] = x[1].sort().values                       # ordered rows
    x[2] = x[2].sort(descending=True).values
    for r, step in ((3, 256), (4, 128), (5, 64)):   # every leader in one thread, in two, in four
        x[r, ::step] = 30 + torch.randn(len(range(0, V, step)), generator=g)
    x[6] = 0.5                                      # one value
    x[7] = torch.randint(0, 3, (V,), generator=g).float()  # three values
    x[8, ::2] = float("-inf")
    x[9] = float("-inf")
    x[9, V // 2] = 1.0
    x[10] = 0.0
    x[10, 1::2] = -0.0
    x[11, V // 3] = 3e38                            # the search's interval spans the format
    x[12] = -x[11].abs()
    x[13] = torch.randn(V, generator=g) * 1e-30
    x[14, :3] = 40.0                                # leaders far above the bulk
    x[15] = x[15] * 100
    return x.to(torch.bfloat16)


@pytest.mark.parametrize("V", [7, 255, 256, 300, 2048, 2049, 4096])
@pytest.mark.parametrize("k", [1, 50, 64, 128, 129, 300])
def test_selection_edges(gpu, V, k):
    from m3x import ops
    logits = _rows(V, V + k)
    B = logits.shape[0]
    u = torch.rand(B, generator=torch.Generator().manual_seed(k))
    out = torch.empty(B, dtype=torch.int32, device=gpu)
    ops.topk_sample(logits.to(gpu), u.to(gpu), 1 / 0.7, k, False, out)
    ref = C.topk_sample_rows(bf16_bits(logits), 1 / 0.7, k, u.numpy())
    assert np.array_equal(out.cpu().numpy(), ref), np.nonzero(out.cpu().numpy() != ref)
    cb0 = torch.zeros(B, dtype=torch.long, device=gpu)
    hist = torch.randint(-1, V, (B, 12), generator=torch.Generator().manual_seed(V))
    hist[:, 3] = hist[:, 4]                         # a code twice in the window takes one penalty
    dev = hist.to(gpu)
    rep = torch.full((B,), 0.8)
    ops.cb0_sample(logits.to(gpu), -1, torch.arange(B, device=gpu), u.to(gpu), temp=0.9, top_k=k, rep_t=rep.to(gpu),
                   hist_t=dev, cb0_out=cb0)
    bits = bf16_bits(logits)
    for b in range(B):
        h = hist[b].numpy().astype(np.int64).copy()
        code, _ = C.cb0_sample(bits[b], -1, 0.9, min(k, V), 0.0, 0.8, h, None, 0, None, None, float(u[b]))
        assert code == int(cb0[b]), b
        assert np.array_equal(dev[b].cpu().numpy(), h)
