"""Mixed steps called eagerly: decode rows and prompt tiles one after the other, or beside each other, give the same bits."""
import numpy as np
import pytest
import torch

from dli_amd import ops
from dli_amd.ops.kv_layout import allocate_kv_cache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("heads,kv_heads", [(32, 8), (8, 1)])
def test_one_after_the_other_and_beside(monkeypatch, dtype, heads, kv_heads):
    decode, prompts = [33, 400, 1], [(70, 70), (300, 260)]                 # contexts; (context with the new tokens, new tokens)
    lens = np.array(decode + [l for l, _ in prompts])
    new = np.array([1] * len(decode) + [n for _, n in prompts])
    pages = (lens + 31) // 32
    g = torch.Generator(device="cuda").manual_seed(5)
    kc, vc = allocate_kv_cache(1, int(pages.sum()) + 1, kv_heads, 128, dtype, "cuda")[0]
    for t in (kc, vc):
        t.copy_(torch.randn(t.shape, generator=g, device="cuda").to(dtype))
    bt = np.zeros((len(lens), int(pages.max())), dtype=np.int32)
    for i, n in enumerate(pages):
        bt[i, :n] = 1 + pages[:i].sum() + np.arange(n)
    cu = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).cuda()
    ts, t0 = ops.build_prefill_tiles(new[len(decode):], len(decode), ops.prefill_tile_tokens(heads, kv_heads), lens[len(decode):])
    meta = ops.AttnMetadata(len(decode), len(prompts), int(new.sum()), None, None, cu(bt), cu(lens), cu(np.concatenate([[0], np.cumsum(new)])),
                            max_seq_len=int(lens.max()), prefill_tile_seq=cu(ts), prefill_tile_q0=cu(t0), num_prefill_tiles=len(ts))
    ops.attach_decode_worklist(meta, lens[:len(decode)], heads, kv_heads, "cuda")
    qkv = torch.randn(int(new.sum()), (heads + 2 * kv_heads) * 128, generator=g, device="cuda", dtype=torch.bfloat16)
    out = []
    for beside in (False, True):
        monkeypatch.setattr(ops, "attention_beside", lambda *a, b=beside: b)
        out += [ops.paged_attention(qkv, kc, vc, meta, heads, kv_heads, 128, 0.088) for _ in range(3)]
    assert all(torch.equal(out[0], o) for o in out[1:]) and bool(torch.isfinite(out[0].float()).all())
