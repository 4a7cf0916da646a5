"""The 256- and 128-row GEMM tiles of four waves (``csrc/kernels/gemm_core.h``) at the edges of their tiles and schedules."""
import pytest
import torch

from dli_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _e4m3_operands(m, n, k, pad=0):
    g = torch.Generator(device=DEV).manual_seed(m * 7919 + n * 31 + k)
    x = torch.randn(m, k, generator=g, device=DEV) * torch.exp(torch.randn(m, 1, generator=g, device=DEV))
    xs = x.abs().amax(1, keepdim=True) / 448.0
    q = torch.empty(m, k + pad, dtype=torch.float8_e4m3fn, device=DEV)[:, :k]
    q.copy_(x / xs)
    wq, ws = ops.quant_weight_fp8(torch.randn(n, k, generator=g, device=DEV) * k ** -0.5)
    return q, xs, wq, ws


# rows around both tile heights; one column block, a last group of column blocks that is not full; more 256-row tiles than compute units, more 128-row
# ones alone and behind them (MANY_HALVES; the last of 640 rows' tiles full, of 1100 and 1570 ragged); the fewest steps, an even number of step pairs,
# an odd one
MANY_HALVES = [(640, 21760, 256), (1100, 26624, 512), (1570, 28160, 768)]


@pytest.mark.parametrize("m,n,k", [(1, 256, 256), (127, 256, 512), (128, 512, 768), (129, 256, 256), (255, 2304, 512), (256, 256, 256),
                                   (257, 768, 768), (383, 2560, 256), (385, 256, 4096), (3000, 7168, 512), (4300, 8192, 256)] + MANY_HALVES)
def test_e4m3_tiles_against_64_bits(m, n, k):
    """Per element: half a bf16 ulp (up to 2^-8 of the value), and 2^-24 of the sum of magnitudes for each of k additions."""
    assert (ops.hip().gemm_e4m3_plan(m, n)[1] > 256) == ((m, n, k) in MANY_HALVES)          # a workgroup's second tile of 128 rows
    q, xs, wq, ws = _e4m3_operands(m, n, k, pad=16 if m % 2 else 0)
    a, b = q.double() * xs.double(), wq.double() * ws.double().t()
    want = a @ b.t()
    bound = 2.0 ** -8 * want.abs() + k * 2.0 ** -24 * (a.abs() @ b.abs().t())
    for out in (None, torch.full((m + 2, n), 7.0, dtype=torch.bfloat16, device=DEV)):
        got = ops.hip().gemm_e4m3(q, xs, wq, ws, None if out is None else out[1:m + 1])
        assert ((got.double() - want).abs() <= bound).all()
        assert out is None or bool((out[0] == 7.0).all() and (out[-1] == 7.0).all())         # rows past the last are not written


def test_e4m3_rule_sends_each_call_to_a_path_that_takes_it():
    """Own tiles and the library on the calls of ``linear_fp8``: odd sizes and strides that the tiles do not take, an out buffer, NaN rows."""
    for m, n, k in ((2000, 4096, 1024), (2000, 4096, 1152), (2000, 4112, 1024), (40, 512, 256)):
        q, xs, wq, ws = _e4m3_operands(m, n, k)
        want = (q.float() * xs) @ (wq.float() * ws.t()).t()
        assert ops._e4m3_ok(q, xs, wq, ws, None) == ((m, n, k) == (2000, 4096, 1024))
        out = torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
        for got in (ops.linear_fp8(None, wq, ws, xq=(q, xs)), ops.linear_fp8(None, wq, ws, xq=(q, xs), out=out)):
            assert (got.float() - want).abs().max() / want.abs().max() < 1e-2
    q, xs, wq, ws = _e4m3_operands(2000, 4096, 1024)
    xs[77] = float("nan")
    got = ops.linear_fp8(None, wq, ws, xq=(q, xs))
    assert bool(got[77].isnan().all()) and not bool(got[:77].isnan().any()) and not bool(got[78:].isnan().any())
