"""Alignment of routed pairs (moe_align_kernel) at its edges: runs of more than 512 pairs a wave, numbers of experts around powers of two, one pair."""
import pytest
import torch

from dli_amd import ops
from dli_amd.ops import reference as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,El,off,k", [(1, 2, 2, 0, 2), (33, 1, 1, 0, 1), (700, 5, 5, 0, 3), (513, 64, 64, 0, 4), (300, 33, 17, 9, 2), (9000, 16, 16, 0, 2)])
@pytest.mark.parametrize("rows", [32, 128])
def test_experts_of_any_number(T, E, El, off, k, rows):
    g = torch.Generator(device="cuda").manual_seed(T + E)
    rnd = lambda *s, scale=1.0: (torch.randn(*s, generator=g, device="cuda") * scale).bfloat16()
    x, logits, w13, w2 = rnd(T, 128), rnd(T, E, scale=2.0), rnd(El, 256, 128, scale=0.1), rnd(El, 128, 128, scale=0.1)
    got = ops.hip().fused_moe(x, logits, w13, w2, k, off, rows).float()
    want = ref.moe_ref(x.float(), logits.float(), w13.float(), w2.float(), k, off).float()
    assert (got - want).abs().max() / want.abs().max() < 3e-2  # bf16 activations between the products and bf16 results
