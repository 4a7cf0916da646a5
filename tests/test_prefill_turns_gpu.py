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
