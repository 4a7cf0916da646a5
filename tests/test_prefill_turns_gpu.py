"""Prefill attention, turns of one and two pages: every number of pages that a turn, a group and a pair of groups can end with."""
import numpy as np
import pytest
import torch

from dli_amd import ops
from dli_amd.ops import reference as ref
from test_kernels_gpu import _bf, _fill_cache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("copies", [1, 40])                        # 96 tiles: two groups; 3840: one
@pytest.mark.parametrize("kv_dtype", [torch.bfloat16, torch.float8_e4m3fn])
def test_page_counts_of_a_turn(kv_dtype, copies):
    """1 to 12 pages, the last of 1 and of 32 tokens (the chunk crosses a page's end), 3 new tokens each.  Weights and results are rounded to bf16
    (half an ulp each: 2^-8 of the value at most, half of that on average; |v| ≤ 4.5 here); e4m3 keys and values enter as they are stored."""
    Hq, Hkv = 16, 4
    seq_lens = [32 * p + e for p in range(12) for e in (4, 32)] * copies
    n = len(seq_lens)
    scales = (0.5, 0.25) if kv_dtype == torch.float8_e4m3fn else (1.0, 1.0)
    kc, vc, bt = _fill_cache(Hq, Hkv, seq_lens, kv_dtype, seed=27, scales=scales)
    qkv = _bf(3 * n, (Hq + 2 * Hkv) * 128, seed=28)
    qkv[::3] *= 8
    i32 = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.int32, device="cuda")
    qsl = i32(np.arange(n + 1) * 3)
    ts, t0 = ops.build_prefill_tiles(np.full(n, 3), 0, ops.prefill_tile_tokens(Hq, Hkv))
    meta = ops.AttnMetadata(num_decode=0, num_prefill=n, num_tokens=3 * n, positions=None, slot_mapping=None, block_tables=bt, seq_lens=i32(seq_lens),
                            query_start_loc=qsl, decode_splits=1, prefill_tile_seq=i32(ts), prefill_tile_q0=i32(t0), num_prefill_tiles=len(ts))
    got = ops.paged_attention(qkv, kc, vc, meta, Hq, Hkv, 128, 0.088, *scales).float()
    want = ref.paged_attention_ref(qkv[:, :Hq * 128].reshape(3 * n, Hq, 128), kc, vc, bt, i32(seq_lens), qsl, 0.088, *scales).float()
    torch.testing.assert_close(got, want, rtol=2 ** -7, atol=2 ** -9 * 4.5)


@pytest.mark.parametrize("first,second", [(5, 40), (40, 5), (5, 70), (9, 20), (130, 170)])
@pytest.mark.parametrize("kv_dtype", [torch.bfloat16, torch.float8_e4m3fn])
def test_largest_weight_of_every_page_is_exact(kv_dtype, first, second):
    """Two tokens carry a row's whole weight, `second` the larger part.  Where it comes in a later page than `first`, both weights are 1 when their pages are
    added; only the result is rounded then: half a bf16 ulp, and 2^-18 for the fp32 exponentials and sums.  Where it does not, `first`'s weight is
    rounded to bf16 too."""
    Hq, Hkv, L, n = 32, 8, 300, 4
    g = torch.Generator().manual_seed(first)
    kc, vc, bt = _fill_cache(Hq, Hkv, [L], kv_dtype, seed=29)
    k, v = torch.zeros(L, Hkv, 128), torch.randn(L, Hkv, 128, generator=g).to(kv_dtype).float()
    k[:, :, 0] = -16.0
    k[first, :, 0], k[second, :, 0] = 1.0, 1.25
    slots = (bt[0, :(L + 31) // 32].long().cpu()[:, None] * 32 + torch.arange(32)[None, :]).reshape(-1)[:L].to(torch.int32).cuda()
    from dli_amd.ops.kv_layout import write_kv_ref
    write_kv_ref(k.bfloat16().cuda(), v.bfloat16().cuda(), slots, kc, vc)
    qkv = torch.zeros(n, (Hq + 2 * Hkv) * 128, dtype=torch.bfloat16)
    x = (2.0 + 8.0 * torch.rand(n, Hq, generator=g)).bfloat16()
    qkv.view(n, -1, 128)[:, :Hq, 0] = x
    i32 = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.int32, device="cuda")
    ts, t0 = ops.build_prefill_tiles(np.array([n]), 0, ops.prefill_tile_tokens(Hq, Hkv))
    meta = ops.AttnMetadata(num_decode=0, num_prefill=1, num_tokens=n, positions=None, slot_mapping=None, block_tables=bt, seq_lens=i32([L]), max_seq_len=L,
                            query_start_loc=i32([0, n]), decode_splits=1, prefill_tile_seq=i32(ts), prefill_tile_q0=i32(t0), num_prefill_tiles=len(ts))
    assert ops.hip().prefill_page_groups(len(ts), Hkv, Hq // Hkv, L, 1, kv_dtype != torch.bfloat16) == 2        # two groups, ten pages
    got = ops.paged_attention(qkv.cuda(), kc, vc, meta, Hq, Hkv, 128, 1.0).double().cpu().view(n, Hq, 128)
    a = torch.exp(-0.25 * x.double())[:, :, None]
    va, vb = (v[t].double().repeat_interleave(Hq // Hkv, 0)[None] for t in (first, second))
    want = (a * va + vb) / (a + 1.0)
    half_ulp = torch.exp2(torch.floor(torch.log2(want.abs().clamp_min(2.0 ** -126))) - 8)
    bound = half_ulp + 2.0 ** -18 * (a * va.abs() + vb.abs()) / (a + 1.0)
    if second // 32 <= first // 32:
        bound = bound + 2.0 ** -8 * a * va.abs() / (a + 1.0)
    assert ((got - want).abs() <= bound).all()
