"""Down projections of routed experts whose last tiles are cut along K (moe.hip, cut_plan): whole rounds in front of them or none, column groups of
other widths, half tiles, fp32 and bf16 rows, experts that live elsewhere."""
import pytest
import torch

from dli_amd import ops
from dli_amd.ops import reference as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,I,E,El,off", [(600, 4096, 4096, 2, 2, 0),       # 96 tiles, no whole round
                                             (2300, 4096, 4096, 2, 2, 0),      # 256 + 32, fp32 rows
                                             (4200, 4096, 2048, 2, 2, 0),      # 512 + 32 of which half are half tiles, bf16 rows
                                             (1000, 512, 4096, 8, 8, 0),       # two column blocks
                                             (3000, 3072, 2048, 2, 2, 0),      # 256 + 32 in a column group of four
                                             (2300, 4096, 2048, 3, 2, 1)])     # pairs of an expert that is not here
def test_cut_tiles_match_reference(T, H, I, E, El, off):
    g = torch.Generator(device="cuda").manual_seed(T + H)
    rnd = lambda *s, scale=1.0: (torch.randn(*s, generator=g, device="cuda") * scale).bfloat16()
    x, logits, w13, w2 = rnd(T, H), rnd(T, E, scale=2.0), rnd(El, 2 * I, H, scale=0.02), rnd(El, H, I, scale=0.02)
    got = ops.hip().fused_moe(x, logits, w13, w2, 2, off, 256).float()
    small = ops.hip().fused_moe(x, logits, w13, w2, 2, off, 128).float()
    want = ref.moe_ref(x.float(), logits.float(), w13.float(), w2.float(), 2, off).float()
    scale = want.abs().max()
    assert torch.isfinite(got).all()
    assert (got - want).abs().max() / scale < 3e-2             # bf16 activations between the products and bf16 results
    assert (got - small).abs().max() / scale < 1.5e-2
    for _ in range(3):                                         # slices are summed in fixed order
        assert torch.equal(ops.hip().fused_moe(x, logits, w13, w2, 2, off, 256).float(), got)
