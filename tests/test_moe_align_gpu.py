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


@pytest.mark.parametrize("T,E,k,near", [(4500, 64, 2, 1), (9000, 64, 2, 64), (9000, 3, 1, 700), (600, 64, 1, 32)])
def test_counts_that_other_lanes_moved_on(T, E, k, near):
    """Neighbouring pairs of one expert, or of one in every 64 and another in the next: each step of a wave goes on from a count that a lane other than the
    present expert's first wrote the step before.  A count read too early puts two pairs into one row and leaves their tokens wrong."""
    g = torch.Generator(device="cuda").manual_seed(T)
    rnd = lambda *s, scale=1.0: (torch.randn(*s, generator=g, device="cuda") * scale).bfloat16()
    x, logits, w13, w2 = rnd(T, 128), rnd(T, E), rnd(E, 256, 128, scale=0.1), rnd(E, 128, 128, scale=0.1)
    logits[torch.arange(T, device="cuda"), torch.arange(T, device="cuda") // near % E] = 12.0
    got = ops.hip().fused_moe(x, logits, w13, w2, k, 0, 32).float()
    want = ref.moe_ref(x.float(), logits.float(), w13.float(), w2.float(), k, 0).float()
    assert (got - want).abs().max() / want.abs().max() < 3e-2  # as above
