"""The cut-off's row maxima and bins (``csrc/kernels/sampler.hip``) on rows where packed comparisons can go wrong."""
import pytest
import torch

from dli_amd import ops
from dli_amd.ops import reference as ref

pytestmark = pytest.mark.gpu

_INF, _LOWEST = float("inf"), torch.finfo(torch.bfloat16).min


def _row(kind, v, g):
    x = torch.randn(v, generator=g) * 3.0
    if kind == "negative":
        x = -x.abs() - 0.5
    elif kind == "all but one masked":
        x, x[v // 3] = torch.full((v,), -_INF), -7.0
    elif kind == "zero is the largest":
        x = torch.where(x > 0, 0.0, -1.0)
    elif kind == "lowest":
        x[::2] = _LOWEST
    elif kind == "far below":
        x[1::3] = -1e9
    elif kind == "one positive among negative":
        x, x[v - 1] = -x.abs() - 1.0, 1e-30
    elif kind == "equal":
        x = torch.full((v,), -2.5)
    return x.bfloat16()


# row lengths: one launch, two launches of four and of sixteen chunks a thread, the last with threads that have none
@pytest.mark.parametrize("v", [2048, 8200, 32000, 128256])
def test_cut_off_rows(v):
    kinds = ["plain", "negative", "all but one masked", "zero is the largest", "lowest", "far below", "one positive among negative", "equal"]
    g = torch.Generator().manual_seed(v)
    rows = torch.stack([_row(k, v, g) for k in kinds for _ in range(3)])
    b = rows.shape[0]
    temp = torch.full((b,), 0.9)
    top_p = torch.tensor([0.92, 1.0, 0.7] * len(kinds))
    top_k = torch.tensor([0, 7, 40] * len(kinds), dtype=torch.int32)
    noise = torch.rand(b, v, generator=g).clamp_min(1e-6)
    out = torch.empty(b, dtype=torch.int64, device="cuda")
    cu = lambda t: t.cuda()
    zeros = torch.zeros(b, dtype=torch.int64, device="cuda")
    ops.hip().sample(out, cu(rows), cu(temp), cu(top_p), cu(top_k), zeros, zeros, cu(noise))
    got = out.cpu()
    for i in range(b):
        x = rows[i].double()
        # ties at the cut-off are all kept: the draw is over every token whose logit reaches the smallest kept one
        z = x / 0.9
        order = torch.sort(z, descending=True).values
        cut = -_INF
        if top_k[i] > 0:
            cut = order[min(int(top_k[i]), v) - 1].item()
        if top_p[i] < 1.0:
            w = torch.exp(order - order[0])
            w[order < cut] = 0.0
            c = torch.cumsum(w, 0) / w.sum()
            cut = max(cut, order[int((c >= float(top_p[i])).nonzero()[0])].item())
        score = z - torch.log(-torch.log(noise[i].double()))
        score[z < cut] = -_INF
        best = score.max()
        assert score[got[i]] >= best - 1e-5 * max(1.0, abs(best.item())), (kinds[i // 3], i % 3)


# rows that every logit draws in: one launch, slices of one and of four chunks a thread; −0, masks and equal logits among them
@pytest.mark.parametrize("b,v", [(3, 8), (5, 8192), (7, 8200), (40, 131072), (520, 32776)])
def test_plain_draws_are_the_row_kernels(b, v):
    """Rows without cut-off draw in a loop of their own, without keys; the fp32 rows' kernel draws each logit that passes its cut-off: same ids."""
    g = torch.Generator().manual_seed(v)
    x = (torch.randn(b, v, generator=g) * torch.tensor([0.0, 0.5, 4.0])[torch.arange(b) % 3, None]).bfloat16()
    x[1, ::2], x[2, v // 2:] = -0.0, -_INF
    i = torch.arange(b)
    temp, ones, none = (0.3 + 0.35 * (i % 5)).cuda(), torch.ones(b).cuda(), torch.zeros(b, dtype=torch.int32).cuda()
    x = x.cuda()
    for r in range(3):
        seeds, steps = (i * 104729 + r).cuda(), (i * 17 + r).cuda()
        assert torch.equal(ops.sample(x, temp, ones, none, seeds, steps), ops.sample(x.float(), temp, ones, none, seeds, steps))
