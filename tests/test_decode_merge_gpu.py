"""The merge of a decode row's ranges (decode_reduce_kernel) at the numbers of ranges where its loop changes, against 64 bits over the same partial results."""
import pytest
import torch

from dli_amd import ops
from dli_amd.ops.kv_layout import allocate_kv_cache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("splits", [2, 8, 9, 16, 17, 32, 33, 48, 49, 64])
def test_ranges_are_added_up(splits, dtype):
    heads, kv_heads, lens = 8, 2, [1500, 31, 900]                # (the short row has empty ranges)
    g = torch.Generator(device="cuda").manual_seed(splits)
    pages = [(n + 31) // 32 for n in lens]
    kc, vc = allocate_kv_cache(1, sum(pages), kv_heads, 128, dtype, "cuda")[0]
    for t in (kc, vc):
        t.copy_(torch.randn(t.shape, generator=g, device="cuda").to(dtype))
    bt = torch.zeros(3, max(pages), dtype=torch.int32, device="cuda")
    for i, n in enumerate(pages):
        bt[i, :n] = torch.arange(sum(pages[:i]), sum(pages[:i + 1]), dtype=torch.int32, device="cuda")
    q = torch.randn(3, heads * 128, generator=g, device="cuda").bfloat16()
    out, ws = torch.empty_like(q), torch.zeros(3 * splits * heads * 130, device="cuda")
    ops.hip().paged_attention_decode(out, q, kc, vc, bt, torch.tensor(lens, dtype=torch.int32, device="cuda"), 3, heads, kv_heads, 0.088, splits, ws, 1.0, 1.0, None)
    o, ml = ws.double()[:3 * splits * heads * 128].view(3, splits, heads, 128), ws.double()[3 * splits * heads * 128:].view(3, splits, heads, 2)
    f = torch.exp2(ml[..., 0] - ml[..., 0].amax(1, keepdim=True))
    want = (f[..., None] * o).sum(1) / (f * ml[..., 1]).sum(1)[..., None]
    # one rounding to bf16 (2^-9); fp32 sums of up to 64 terms and the fast exponential stay far below it
    torch.testing.assert_close(out.view(3, heads, 128).double(), want, rtol=2 ** -8, atol=1e-5)
