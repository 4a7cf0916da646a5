"""Mixed steps whose decode rows and prompt tiles have launches of their own (DLI_ATTN_ONE_LAUNCH=0, or where the rule for one launch says so): one after the
other, beside each other on two streams, and in one launch they give the same bits."""
import numpy as np
import pytest
import torch

from dli_amd import ops
from dli_amd.ops import reference as ref
from dli_amd.ops.kv_layout import allocate_kv_cache
from test_mixed_launch_gpu import _step

pytestmark = pytest.mark.gpu


class _Counted:
    """A kernel's op that remembers on which stream it was launched."""

    def __init__(self, name):
        self.name, self.op, self.streams = name, getattr(ops.hip(), name), []

    def __call__(self, *a):
        self.streams.append(torch.cuda.current_stream())
        return self.op(*a)


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
    out, asked, prefill, one = [], [], _Counted("paged_attention_prefill"), _Counted("paged_attention_mixed")
    monkeypatch.setattr(ops, "ONE_LAUNCH_ATTN", False)
    monkeypatch.setattr(ops.hip(), prefill.name, prefill, raising=False)
    monkeypatch.setattr(ops.hip(), one.name, one, raising=False)
    for beside in (False, True):
        monkeypatch.setattr(ops, "attention_beside", lambda *a, b=beside: asked.append(b) or b)
        out += [ops.paged_attention(qkv, kc, vc, meta, heads, kv_heads, 128, 0.088) for _ in range(3)]
    main = torch.cuda.current_stream()
    assert asked == [False] * 3 + [True] * 3 and not one.streams
    assert [s == main for s in prefill.streams] == [True] * 3 + [False] * 3
    # one launch of two page groups, whose rows have as many waves as in their own: the same sums in the same order
    monkeypatch.setattr(ops, "ONE_LAUNCH_ATTN", True)
    out.append(ops.paged_attention(qkv, kc, vc, meta, heads, kv_heads, 128, 0.088))
    assert len(one.streams) == 1 and len(prefill.streams) == 6
    assert all(torch.equal(out[0], o) for o in out[1:]) and bool(torch.isfinite(out[0].float()).all())


def test_launches_of_their_own_where_the_rule_says_so(monkeypatch):
    """Two short decode rows beside a prompt of 1100 tokens behind 623, whose own launch takes two page groups past 256 tiles."""
    kc, vc, meta, qkv = _step(32, 8, torch.bfloat16, [33, 400], [(1723, 1100)])
    prefill, one = _Counted("paged_attention_prefill"), _Counted("paged_attention_mixed")
    monkeypatch.setattr(ops.hip(), prefill.name, prefill, raising=False)
    monkeypatch.setattr(ops.hip(), one.name, one, raising=False)
    got = ops.paged_attention(qkv, kc, vc, meta, 32, 8, 128, 0.088).float()
    assert len(prefill.streams) == 1 and not one.streams
    T = qkv.shape[0]
    want = ref.paged_attention_ref(qkv[:, :4096].reshape(T, 32, 128), kc, vc, meta.block_tables, meta.seq_lens, meta.query_start_loc, 0.088).float()
    torch.testing.assert_close(got, want, rtol=2e-2, atol=2e-2)      # (both round to bf16; the weights are bf16 in the products)
