"""Rows past 256 with long K: the rule that sends them to sliced own tiles, at sizes timed both ways, and the products at its edges."""
import pytest
import torch

from dli_amd import ops
from test_dispatch import _Recorder


def test_sizes_on_both_sides_of_the_line():
    f = ops.tile_slices
    assert [f(*s) for s in ((257, 4096, 14336), (512, 4096, 14336), (768, 4096, 14336), (1024, 4096, 14336), (2048, 4096, 14336), (512, 8192, 28672),
                            (512, 2048, 28672), (1024, 1024, 14336))] == [8, 8, 5, 4, 2, 4, 8, 8]
    assert [f(*s, True) for s in ((257, 7168, 8192), (768, 7168, 8192), (1024, 7168, 8192), (1024, 3584, 8192))] == [4, 3, 2, 4]
    assert not any(f(*s) for s in ((256, 4096, 14336), (2049, 4096, 14336), (700, 8192, 28672), (512, 8192, 8192), (1024, 4096, 4096), (257, 1024, 14336),
                                   (512, 4096, 14336 + 32), (512, 4000, 14336), (512, 0, 14336), (0, 4096, 14336), (512, 7168, 8192), (512, 7168, 4096, True)))


def test_wide_weights_and_half_empty_row_tiles():
    """Two or three slices lose to the library where the last row tile is nearly empty (16384 × 16384 at 257 rows 178 µs / 213), four do not."""
    f = ops.tile_slices
    assert not any(f(*s) for s in ((257, 16384, 16384), (400, 16384, 16384), (310, 13824, 18240), (569, 10496, 13504), (257, 10240, 16384), (300, 9728, 15616)))
    assert not any(f(*s, True) for s in ((257, 16384, 7680), (315, 15616, 11648), (257, 10240, 8576)))
    assert [f(*s) for s in ((512, 16384, 16384), (1024, 8192, 14336), (330, 10240, 14336), (257, 8192, 14336), (257, 7168, 18432))] == [2, 2, 3, 4, 4]
    assert [f(*s, True) for s in ((512, 16384, 16384), (330, 10240, 8576), (257, 8192, 8576), (257, 7168, 8192))] == [2, 3, 4, 4]
    assert not any(f(*s, True) for s in ((345, 8192, 8192), (512, 16384, 8192)))       # (at this K the wide ones are no faster however full)


def test_long_enough_sums():
    """K on both sides of the lines, at sizes that are no preset's: below them the library wins at some sizes."""
    f = ops.tile_slices
    assert [f(512, 4096, k) > 0 for k in (9216, 11008, 12224, 12288, 13824)] == [False, False, False, True, True]
    assert [f(512, 5120, k, True) > 0 for k in (5120, 6144, 7104, 7168, 9216)] == [False, False, False, True, True]


def test_gate_up_goes_to_the_library_where_the_switch_says_so(monkeypatch):
    """DLI_NO_GEMM256_SWIGLU=1 names every untuned gate/up product on the own 256² tiles, the sliced ones too; down projections are none of its business."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    monkeypatch.setattr(ops, "hip", _Recorder)
    monkeypatch.setattr(ops, "_plain", lambda *t: True)

    def route(f, m, n, k):
        with FakeTensorMode(), pytest.raises(RuntimeError) as e:
            f(*(torch.empty(r, k, device="cuda", dtype=torch.bfloat16) for r in (m, n)))
        return str(e.value)
    sizes = ((512, 7168, 8192), (300, 7168, 12288), (700, 28672, 4096))
    assert [route(ops.linear_swiglu, *s) for s in sizes] == ["dense_gemm256"] * 3
    monkeypatch.setattr(ops, "GEMM256_SWIGLU", False)
    assert [route(ops.linear_swiglu, *s) for s in sizes] == ["silu_and_mul"] * 3
    assert route(ops.linear, 512, 4096, 14336) == "dense_gemm256"


def test_short_products_keep_their_last_round_whole():
    """K timed with the last round cut and whole, on both sides of the line."""
    assert not any(ops.swiglu_tail_cut(k) for k in (512, 1024, 2048, 2560))
    assert all(ops.swiglu_tail_cut(k) for k in (3072, 4096, 8192))


@pytest.mark.gpu
@pytest.mark.parametrize("k", [512, 3072])
def test_last_round_of_the_untuned_gate_up(monkeypatch, k):
    """300 tiles: a whole round and 44 more, whole behind a short K, in slices behind a long one.  Against fp32 products; and the call is asked for as the line says."""
    asked, op = [], ops.hip().dense_gemm256
    monkeypatch.setattr(ops.hip(), "dense_gemm256", lambda x, w, *a: (asked.append(a[-1]), op(x, w, *a))[1], raising=False)
    g = torch.Generator(device="cuda").manual_seed(k)
    x = torch.randn(730, k, generator=g, device="cuda").bfloat16()
    w = (torch.randn(25600, k, generator=g, device="cuda") * k ** -0.5).bfloat16()
    got, y = ops.linear_swiglu(x, w).float(), x.float() @ w.float().t()
    torch.testing.assert_close(got, torch.nn.functional.silu(y[:, :12800]) * y[:, 12800:], rtol=2 ** -7, atol=2e-2)      # as below
    assert asked == [k >= 3072]


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,swiglu", [(257, 1024, 14336, False), (1025, 1024, 14336, False), (520, 4096, 14336, False), (300, 7168, 8192, True),
                                          (769, 3584, 8192, True)])
def test_products_match_fp32(m, n, k, swiglu):
    g = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(m, k, generator=g, device="cuda").bfloat16()
    w = (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).bfloat16()
    got = (ops.linear_swiglu(x, w) if swiglu else ops.linear(x, w)).float()
    want = x.float() @ w.float().t()
    if swiglu:
        want = torch.nn.functional.silu(want[:, :n // 2]) * want[:, n // 2:]
    torch.testing.assert_close(got, want, rtol=2 ** -7, atol=2e-2)      # one rounding to bf16 (and the fast exponential); sums of K products in fp32
