"""Rules that choose a kernel, as far as they run without a GPU."""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from dli_amd import ops

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _moe_rows(env, *args):
    code = f"from dli_amd import ops; print(*[ops.hip().moe_tile_rows(*a) for a in {args!r}])"
    e = {**os.environ, **env}
    return [int(x) for x in subprocess.run([sys.executable, "-c", code], cwd=ROOT, env=e, capture_output=True, text=True, check=True).stdout.split()]


@pytest.mark.parametrize("asked", ["96", "-5", "128"])
def test_expert_row_tiles_are_ones_that_a_kernel_has(asked):
    """The experts' GEMMs align rows to this number and launch the tile of that size: any other value would be tiles past the rows."""
    H = 4096
    calls = (0, 8, H, True), (0, 4000, H, True), (0, 4000, H, False), (32, 4000, H, True), (64, 8, H, True), (256, 8, H, True), (256, 8, H, False)
    assert _moe_rows({"DLI_MOE_TILE": asked}, *calls) == [128, 128, 128, 32, 64, 256, 128]


@pytest.mark.parametrize("hidden", [512, 1920, 2048, 4096])
def test_expert_row_tiles_by_rows_and_by_choice(hidden):
    """Up to 53 rows the streaming tiles, from 128 the 256² ones where they fit; between the two those of 256 rows only for wide layers."""
    rule = ops.hip().moe_tile_rows
    between = 256 if hidden >= 2048 else 128
    for rows, want in ((0, 32), (1, 32), (20, 32), (21, 64), (53, 64), (54, between), (127, between), (128, 256), (10 ** 6, 256)):
        assert rule(0, rows, hidden, True) == want and rule(0, rows, hidden, False) == min(want, 128)
        for given in (32, 64, 128, 48, 7, -1):
            assert rule(given, rows, hidden, True) == (given if given in (32, 64) else 128)
        assert rule(256, rows, hidden, True) == 256 and rule(256, rows, hidden, False) == 128


@pytest.mark.parametrize("n,k,plain,swiglu", [
    # rows 17, 32, 33, 64, 65, 128, 129, 192, 256, 257; 1: the streaming tiles
    (4096, 14336, "1111111110", "1111111110"), (4096, 8192, "0011111110", "0011111110"), (6144, 6144, "1111111110", "1111111110"),
    (6144, 4096, "0000000000", "0000000000"), (8192, 4096, "0000000110", "1111110110"), (8192, 8192, "1111111110", "1111111110"),
    (10240, 4096, "0000000000", "1111110000"), (10240, 8192, "1111110000", "1111110000"), (12288, 4096, "0000000000", "0000000000"),
    (16384, 4096, "0000000000", "0000000000"), (16512, 4096, "1111000000", "1111110000"), (24576, 2048, "1111110000", "1111110000"),
    (128256, 4096, "1111110000", "1111110000"), (8192, 28672, "1111111110", "1111111110"), (4097, 14336, "0000000000", "0000000000"),
    (4096, 14400, "1111111110", "1111111110"), (4096, 14337, "0000000000", "0000000000"), (36864, 4096, "1111000000", "1111000000"),
    (45056, 4096, "1111110000", "1111110000"), (36864, 7168, "0000000000", "0000000000"), (57344, 8192, "1111110000", "1111110000"),
    (65536, 5120, "1111000000", "1111000000"), (73728, 7168, "0000000000", "0000000000"), (98304, 7168, "1111110000", "1111110000"),
    (32768, 5120, "1111110000", "1111110000")])
def test_shapes_of_the_streaming_tiles(n, k, plain, swiglu):
    rows = (17, 32, 33, 64, 65, 128, 129, 192, 256, 257)
    assert "".join(str(int(ops.stream_rows_ok(m, n, k))) for m in rows) == plain
    assert "".join(str(int(ops.stream_rows_ok(m, n, k, True))) for m in rows) == swiglu
    assert not ops.stream_rows_ok(0, n, k)


@pytest.mark.parametrize("n,k,plain,swiglu", [
    # rows 144, 160, 193, 208, 224, 248: two row tiles, where the library is slow at whole 32 rows
    (8192, 4096, "000010", "011111"), (8192, 4608, "000010", "111111"), (6144, 5632, "110010", "111111"), (5120, 7168, "111111", "111111"),
    (8192, 7168, "111111", "111111"), (6144, 16384, "111111", "111111"), (4096, 8192, "111111", "111111"), (10240, 8192, "000000", "000000")])
def test_shapes_of_the_streaming_tiles_in_two_row_tiles(n, k, plain, swiglu):
    rows = (144, 160, 193, 208, 224, 248)
    assert "".join(str(int(ops.stream_rows_ok(m, n, k))) for m in rows) == plain
    assert "".join(str(int(ops.stream_rows_ok(m, n, k, True))) for m in rows) == swiglu


class _Recorder:
    """Stands in for the kernels: says which one a call came to."""

    def __getattr__(self, name):
        def call(*a):
            raise RuntimeError(name)
        return call


def test_large_linear_layers_of_decode_batches_under_traces_and_transforms(monkeypatch):
    """The streaming tiles take addresses, so only ordinary tensors go there; fake ones (shape propagation, export) stay with the library
    operation at every row count, as they always did."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    monkeypatch.setattr(ops, "hip", _Recorder)
    with FakeTensorMode():
        w = torch.empty(8192, 8192, device="cuda", dtype=torch.bfloat16)
        for m in (17, 40, 128, 200, 256, 320):
            x = torch.empty(m, 8192, device="cuda", dtype=torch.bfloat16)
            assert ops.stream_rows_ok(m, 8192, 8192) == (m <= 256) and not ops._stream_ok(x, w)
            assert ops.linear(x, w).shape == (m, 8192)
            with pytest.raises(RuntimeError, match="silu_and_mul"):        # (the library's product, then the activation kernel)
                ops.linear_swiglu(x, w)


def test_the_plan_goes_before_the_rule(monkeypatch):
    """A tuned entry decides also where the rule has an opinion; without one, and past the rows that a streaming entry can serve, the rule does."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from dli_amd.ops import gemm_plan
    monkeypatch.setattr(ops, "hip", _Recorder)
    monkeypatch.setattr(ops, "_plain", lambda *t: True)
    plan = gemm_plan.GemmPlan()
    monkeypatch.setattr(ops, "_PLAN", plan)
    n, k = 8192, 8192

    def route(m, swiglu, bias=None):
        x, w = (torch.empty(r, k, device="cuda", dtype=torch.bfloat16) for r in (m, n))
        try:
            return "lib" if (ops.linear_swiglu(x, w) if swiglu else ops.linear(x, w, bias)) is not None else None
        except RuntimeError as e:
            return {"silu_and_mul": "lib"}.get(str(e), str(e))
    with FakeTensorMode():
        for swiglu in (False, True):
            plan.load({})
            assert [route(m, swiglu) for m in (40, 100, 256, 300)] == ["stream_gemm"] * 3 + ["lib"]
            for value, kernel in ((0, "lib"), (4, "dense_gemm256"), (gemm_plan.TAIL, "dense_gemm256"), (gemm_plan.STREAM, "stream_gemm")):
                plan.load({f"{n},{k},{int(swiglu)}": {"128": value}})
                assert [route(m, swiglu) for m in (100, 128, 200)] == [kernel] * 3
                assert route(40, swiglu) == "stream_gemm"                     # below the rows that are tuned
                assert route(300, swiglu) == ("lib" if value == gemm_plan.STREAM else kernel)
        assert route(100, False, torch.empty(n, device="cuda", dtype=torch.bfloat16)) == "lib"
    assert [gemm_plan.STREAM in plan.candidates(m, n, k, False) for m in (65, 256, 257)] == [True, True, False]
    assert plan.load(plan.export()) is None and plan.splits_for(128, n, k, True) == gemm_plan.STREAM


@pytest.mark.parametrize("new,ctx,n,G,form,e4m3", [
    # 8 kv heads of 4 (32-token tiles) or one of 8 (16-token tiles); timed with one page group, two in rounds, two of which the last share: 1, 2, 3
    (64, 0, 4, 4, 1, 1), (200, 0, 4, 4, 1, 1), (256, 0, 4, 4, 2, 2), (16, 1000, 32, 4, 2, 2), (128, 1000, 8, 4, 2, 2), (1000, 0, 1, 4, 2, 2),
    (2000, 0, 2, 8, 2, 2), (17, 0, 37, 4, 1, 1), (100, 0, 16, 4, 1, 1), (128, 1000, 9, 4, 1, 1), (300, 0, 6, 4, 1, 1), (600, 0, 3, 4, 1, 1),
    (400, 1000, 3, 4, 1, 1), (1000, 1000, 2, 4, 1, 1), (16, 1000, 300, 8, 1, 1), (600, 3000, 2, 4, 1, 1), (128, 200, 10, 4, 1, 1),
    (300, 0, 4, 4, 3, 3), (600, 0, 2, 4, 3, 3), (600, 600, 2, 4, 3, 3), (1100, 500, 1, 4, 3, 3), (1300, 300, 1, 4, 3, 3), (2000, 0, 3, 8, 3, 3),
    (1500, 500, 4, 8, 2, 3), (2000, 0, 1, 4, 2, 2), (2048, 0, 1, 4, 2, 2), (2000, 2000, 1, 4, 1, 1), (2049, 0, 1, 4, 1, 1), (100, 0, 40, 4, 1, 1),
    (4000, 0, 1, 4, 1, 1)])
def test_prefill_page_groups(new, ctx, n, G, form, e4m3):
    """Two groups of waves a tile where the chip takes all tiles at once, or where those that share or wait are short ones."""
    heads, tile = (8, 32) if G == 4 else (1, 16)
    tiles = n * ((new + tile - 1) // tile)
    rule = ops.hip().prefill_page_groups
    assert [rule(tiles, heads, G, new + ctx, n, f) for f in (False, True)] == [form, e4m3]
    assert rule(tiles, heads, G, 0, 0, False) == (2 if tiles * heads <= 256 else 1)        # lengths not known


def test_every_prefill_tile_is_taken_once():
    """What a workgroup of two groups takes where the last of them share (``units`` of them), for every number of tiles."""
    units = 256
    for items in range(1, 2 * units + 1):
        over = max(items - units, 0)
        taken = [b + g * over for b in range(items - over) for g in ((0, 1) if b >= units - over else (0,))]
        assert sorted(taken) == list(range(items))


def test_convolution_runs_where_they_fill_the_chip():
    """Sizes timed with a workgroup a token and a workgroup a run of tokens: a step of few channels needs more rows."""
    by_runs = ops.hip().rm_conv_by_runs
    assert all(by_runs(*size) for size in ((128, 4096), (200, 2304), (700, 1024), (2000, 256), (3162, 16384), (128, 3072)))
    assert not any(by_runs(*size) for size in ((127, 8192), (17, 16384), (200, 1024), (1232, 256), (128, 3068)))


def test_plain_tensors():
    import torch.autograd.forward_ad as fw
    t, seen = torch.zeros(4, 4), []
    assert ops._plain(t) and ops._plain(t, torch.nn.Parameter(t, requires_grad=False))
    with torch.no_grad():
        assert ops._plain(torch.nn.Parameter(t))
    with torch.enable_grad():
        assert not ops._plain(t, torch.nn.Parameter(t))
    look = lambda a: seen.append(ops._plain(a)) or a * 1
    torch.func.vmap(look)(t)
    torch.func.jvp(look, (t,), (t,))
    torch.func.grad(lambda a: look(a).sum())(t)
    with fw.dual_level():
        look(fw.make_dual(t, t))
    torch.jit.trace(look, (t,), check_trace=False)
    assert seen == [False] * 5 and ops._plain(t)


@pytest.mark.parametrize("dtype,plain", [(torch.float16, False), (torch.bfloat16, True)])
def test_autocast_to_another_type_is_the_librarys(dtype, plain):
    """``torch.nn.functional.linear`` casts its operands there and returns that type; a kernel would return bf16."""
    before = torch.is_autocast_enabled("cuda"), torch.get_autocast_dtype("cuda")
    try:
        torch.set_autocast_enabled("cuda", True)
        torch.set_autocast_dtype("cuda", dtype)
        assert ops._plain(torch.ones(2, 2, dtype=torch.bfloat16)) is plain
    finally:
        torch.set_autocast_enabled("cuda", before[0])
        torch.set_autocast_dtype("cuda", before[1])


@pytest.mark.gpu
def test_long_sums_under_autocast():
    x, w = torch.ones(512, 14336, device="cuda", dtype=torch.bfloat16), torch.ones(4096, 14336, device="cuda", dtype=torch.bfloat16) / 64
    assert ops.tile_slices(512, 4096, 14336) and ops.linear(x, w).dtype == torch.bfloat16
    with torch.autocast("cuda", dtype=torch.float16):
        assert ops.linear(x, w).dtype == torch.nn.functional.linear(x, w).dtype == torch.float16


def test_short_decode_rows_stay_whole():
    """Sizes timed with rows cut into ranges and whole: (rows, heads, pages of the longest) on both sides of the line."""
    cut = lambda n, heads, pages: len(ops.build_decode_work(np.full(n, 32 * pages), heads)[1]) > 0
    assert not any(cut(*size) for size in ((1, 8, 12), (1, 1, 12), (16, 8, 18), (32, 8, 24), (60, 8, 36), (250, 1, 24), (64, 8, 64)))
    assert all(cut(*size) for size in ((1, 8, 13), (1, 1, 20), (8, 8, 20), (16, 8, 25), (32, 8, 50), (60, 8, 48)))


def test_mixed_attention_takes_a_second_stream_where_it_pays():
    """Sizes timed both ways: (decode rows, longest context, prefill tiles, prompts, heads, kv heads, bytes of a page element)."""
    def beside(rows, longest, tiles, prompts, heads, kv_heads, size):
        meta = ops.AttnMetadata(rows, prompts, 0, None, None, None, None, None, max_seq_len=longest, num_prefill_tiles=tiles)
        return ops.attention_beside(meta, heads, kv_heads, size)
    assert all(beside(*size) for size in ((400, 1500, 66, 3, 32, 8, 1), (200, 1500, 66, 3, 32, 8, 2), (400, 1500, 94, 1, 64, 8, 2),
                                          (96, 1490, 37, 2, 32, 8, 2), (60, 1490, 43, 2, 64, 8, 2), (400, 0, 94, 3, 32, 8, 2)))
    assert not any(beside(*size) for size in ((2, 400, 2, 1, 32, 8, 1), (96, 1490, 37, 2, 32, 8, 1), (200, 1500, 66, 3, 32, 8, 1),
                                              (64, 1318, 65, 3, 32, 8, 2), (64, 994, 76, 4, 32, 8, 2), (200, 999, 51, 4, 64, 8, 1), (400, 1500, 47, 1, 32, 8, 2), (400, 1500, 94, 1, 8, 1, 2), (1, 0, 2, 1, 32, 8, 2)))


def test_slices_of_decode_rows_by_length():
    """Sizes timed whole and cut: (rows, heads, key heads, key width, pages) and the slices that were no slower than another number."""
    slices = lambda *size: ops.hip().sm_head_decode_splits(*size)
    # short rows of 257 … 511 workgroups stay whole whatever the group, and any that has a page alone
    assert [slices(r, h, g, 128, 4) for r, h, g in ((250, 16, 2), (256, 16, 2), (300, 8, 1), (511, 8, 1), (50, 64, 8), (63, 32, 8), (500, 16, 2))] == [1] * 7
    assert [slices(*s) for s in ((250, 16, 2, 128, 13), (250, 32, 2, 256, 64), (120, 16, 4, 256, 64), (128, 32, 8, 128, 64), (1, 32, 8, 128, 1))] == [1] * 5
    # long ones are cut
    assert [slices(*s) for s in ((140, 16, 2, 128, 16), (300, 8, 1, 128, 32), (40, 32, 8, 128, 32), (250, 16, 2, 128, 32), (511, 8, 1, 128, 63), (140, 32, 2, 256, 32))] == [3, 3, 3, 2, 2, 2]
    # no more slices than pages
    assert [slices(1, 32, 1, 576, p) for p in (7, 13, 63)] == [7, 13, 16] and slices(8, 32, 8, 128, 22) == 16
