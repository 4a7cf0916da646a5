"""Mixed steps in one launch (paged_mixed_kernel): octets of workgroups that the tiles or rows do not fill, tiles and rows in turns, both page groups,
work lists and uniform splits, launches of bounds."""
import numpy as np
import pytest
import torch

from dli_amd import ops
from dli_amd.ops import reference as ref
from dli_amd.ops.kv_layout import allocate_kv_cache

pytestmark = pytest.mark.gpu


def _i32(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).cuda()


def _step(heads, kv_heads, dtype, decode, prompts, listed=True, bounds=False, seed=3, extra=40, items=700):
    lens = np.array(decode + [length for length, _ in prompts])
    new = np.array([1] * len(decode) + [n for _, n in prompts])
    pages = (lens + 31) // 32
    g = torch.Generator(device="cuda").manual_seed(seed)
    kc, vc = allocate_kv_cache(1, int(pages.sum()) + 1, kv_heads, 128, dtype, "cuda")[0]
    for t in (kc, vc):
        t.copy_(torch.randn(t.shape, generator=g, device="cuda").to(dtype))
    bt = np.zeros((len(lens), int(pages.max())), dtype=np.int32)
    for i, n in enumerate(pages):
        bt[i, :n] = 1 + pages[:i].sum() + np.arange(n)
    ts, t0 = ops.build_prefill_tiles(new[len(decode):], len(decode), ops.prefill_tile_tokens(heads, kv_heads), lens[len(decode):])
    meta = ops.AttnMetadata(len(decode), len(prompts), int(new.sum()), None, None, _i32(bt), _i32(lens), _i32(np.concatenate([[0], np.cumsum(new)])),
                            max_seq_len=int(lens.max()), prefill_tile_seq=_i32(ts), prefill_tile_q0=_i32(t0), num_prefill_tiles=len(ts))
    if listed:
        ops.attach_decode_worklist(meta, lens[:len(decode)], heads, kv_heads, "cuda", launch_items=items if bounds else 0)
    else:
        meta.decode_splits = 3
        meta.decode_workspace = torch.empty(len(decode) * heads * 3 * 130, dtype=torch.float32, device="cuda")
    if bounds:                                              # what a captured step launches: more tiles than there are, their number on the device
        meta.prefill_tile_seq, meta.prefill_tile_q0 = _i32(np.concatenate([ts, np.zeros(extra)])), _i32(np.concatenate([t0, np.zeros(extra)]))
        meta.num_prefill_tiles, meta.counts_on_device = len(ts) + extra, True
    qkv = torch.randn(int(new.sum()), (heads + 2 * kv_heads) * 128, generator=g, device="cuda", dtype=torch.bfloat16)
    return kc, vc, meta, qkv


ROWS = [1, 33, 700, 65, 32]
CASES = {                                                   # … and the page groups that the rule takes, bf16 and e4m3
    "two groups": (32, 8, ROWS, [(500, 300), (70, 70)], (2, 2)),
    "two groups, few workgroups": (8, 1, ROWS, [(900, 33)], (2, 2)),
    "three key heads": (12, 3, ROWS * 12, [(90, 90), (33, 17)], (2, 2)),
    "three key heads, many rows": (12, 3, ROWS * 100, [(90, 90), (33, 17)], (1, 2)),
    "one head a group": (5, 5, [40], [(40, 40)], (2, 2)),
    "turns, few rows": (32, 8, ROWS, [(2100, 2100)], (1, 1)),
    "turns, many rows": (32, 8, ROWS * 60, [(600, 600)] * 4, (1, 1)),
    "more rows than tiles": (32, 8, ROWS * 40, [(17, 17)], (1, 2)),
}


@pytest.mark.parametrize("form", ["list", "splits", "bounds"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("name", list(CASES))
def test_mixed_launch_matches_reference(monkeypatch, name, dtype, form):
    heads, kv_heads, decode, prompts, groups = CASES[name]
    kc, vc, meta, qkv = _step(heads, kv_heads, dtype, decode, prompts, form != "splits", form == "bounds")
    fp8 = dtype != torch.bfloat16
    if form == "list":
        assert ops.hip().mixed_page_groups(meta.num_prefill_tiles, kv_heads, heads // kv_heads, meta.max_seq_len, meta.num_prefill, meta.num_decode,
                                           fp8) == groups[fp8]
    monkeypatch.setattr(ops, "attention_in_one_launch", lambda *a: True)
    T = qkv.shape[0]
    out = torch.full((T, heads * 128), float("nan"), dtype=torch.bfloat16, device="cuda")
    got = ops.paged_attention(qkv, kc, vc, meta, heads, kv_heads, 128, 0.088, out=out).float()
    want = ref.paged_attention_ref(qkv[:, :heads * 128].reshape(T, heads, 128), kc, vc, meta.block_tables, meta.seq_lens, meta.query_start_loc, 0.088).float()
    torch.testing.assert_close(got, want, rtol=2e-2, atol=2e-2)      # (both round to bf16; the weights are bf16 in the products)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("extra,items", [(0, 100), (60, 2000), (700, 100), (700, 2000)])
@pytest.mark.parametrize("empty", ["", "rows", "tiles", "both"])
def test_bounds_far_from_the_step(dtype, extra, items, empty):
    """A captured launch deals the tiles and rows that there are, by the numbers on the device: grids of many times as many, steps without rows or tiles."""
    decode = ROWS * 2
    kc, vc, meta, qkv = _step(32, 8, dtype, decode, [(300, 290), (90, 17)], True, True, extra=extra, items=items)
    T, nd = qkv.shape[0], len(decode)
    want = ref.paged_attention_ref(qkv[:, :4096].reshape(T, 32, 128), kc, vc, meta.block_tables, meta.seq_lens, meta.query_start_loc, 0.088).float()
    if empty in ("rows", "both"):
        meta.counts[:2] = 0
    if empty in ("tiles", "both"):
        meta.counts[2] = 0
    out = torch.full((T, 4096), float("nan"), dtype=torch.bfloat16, device="cuda")
    got = ops.paged_attention(qkv, kc, vc, meta, 32, 8, 128, 0.088, out=out).float()
    for part, left_out in ((slice(0, nd), empty in ("rows", "both")), (slice(nd, T), empty in ("tiles", "both"))):
        if left_out:
            assert bool(torch.isnan(got[part]).all())
        else:
            torch.testing.assert_close(got[part], want[part], rtol=2e-2, atol=2e-2)      # as above


def test_mixed_launch_replayed_from_a_graph():
    kc, vc, meta, qkv = _step(32, 8, torch.bfloat16, ROWS * 8, [(600, 600), (90, 90)], True, True)
    eager = ops.paged_attention(qkv, kc, vc, meta, 32, 8, 128, 0.088)
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(graph, stream=side, capture_error_mode=ops.CAPTURE_MODE):
        out = ops.paged_attention(qkv, kc, vc, meta, 32, 8, 128, 0.088)
    for seed in range(3):
        qkv.copy_(torch.randn(qkv.shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda", dtype=torch.bfloat16))
        eager = ops.paged_attention(qkv, kc, vc, meta, 32, 8, 128, 0.088)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


def test_separate_launches_where_the_rule_says_so():
    f = lambda tiles, longest, rows: ops.hip().mixed_page_groups(tiles, 8, 4, longest, 1, rows, False)
    assert f(35, 1723, 2) == 0 and f(35, 1723, 100) == 1 and f(25, 1300, 4) == 2 and f(35, 0, 2) == 1
