"""How the e4m3 tiles are dealt to workgroups (``csrc/kernels/gemm_e4m3.hip``): every tile once, and the cost that the plan names is that of the
workgroup with most to do.  Arithmetic only: no GPU."""
import pytest
import torch

from dli_amd import ops

HALF, CUS = 0.58, 256


def _places(total, grid, back):
    """``gcore::Places``: the places of every workgroup's tiles."""
    per, groups, out = -(-total // 8), grid // 8, []
    for block in range(grid):
        x, i = block & 7, block >> 3
        i = groups - 1 - i if back else i
        mine = min(per, total - x * per) - i
        out.append([x * per + i + j * groups for j in range(-(-mine // groups) if mine > 0 else 0)])
    return out


def _rounds(whole, halves):
    grid = min(CUS, -(-whole // 8) * 8 + -(-halves // 8) * 8)
    a, b = _places(whole, grid, False), _places(halves, grid, True)
    assert sorted(sum(a, [])) == list(range(whole)) and sorted(sum(b, [])) == list(range(halves))
    return max(len(p) + HALF * len(q) for p, q in zip(a, b)), grid


SIZES = [(m, n) for n in (256, 2304, 4096, 6144, 8192, 10240, 14336, 28672) for m in (1, 128, 129, 256, 385, 513, 640, 1025, 1152, 1300, 1664, 2000, 2688, 3200, 3456, 4096)]


@pytest.mark.parametrize("m,n", SIZES)
def test_plan_costs_what_its_workgroups_do(m, n):
    whole, halves, grid, rounds = ops.hip().gemm_e4m3_plan(m, n)
    units, cols = -(-m // 128), n // 256
    total, odd = units // 2 * cols, units % 2 * cols
    assert 2 * whole + halves == units * cols
    assert (rounds, grid) == (pytest.approx(_rounds(whole, halves)[0]), _rounds(whole, halves)[1])
    # never the slower of the two forms: all 256-row tiles kept, or those beyond the last whole round cut in two
    rest = total % CUS
    assert rounds == pytest.approx(min(_rounds(total, odd)[0], _rounds(total - rest, 2 * rest + odd)[0]))
    assert ops.hip().gemm_e4m3_fill(m, n) == pytest.approx(m * n / (256 * 256 * CUS * rounds))


# the longest K at which half of the chip is enough, and the fills around the two lines (the last three: more than one round)
@pytest.mark.parametrize("m,n,k,own", [(1280, 4096, 4096, True), (1152, 4096, 4096, False), (1280, 4096, 4352, False), (1408, 4096, 14336, False), (1536, 4096, 14336, False),
                                       (1600, 4096, 14336, True), (768, 8192, 8192, False), (512, 10240, 8192, False), (640, 10240, 8192, True),
                                       (2176, 4096, 14336, True), (1025, 8192, 8192, True), (640, 28672, 4096, True)])
def test_half_filled_rounds_go_where_they_are_faster(m, n, k, own):
    assert ops._e4m3_tiles_pay(m, n, k) == own


def test_only_plain_tensors_and_whole_numbers_reach_the_rule():
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.proxy_tensor import make_fx
    m, n, k = 2000, 4096, 256
    q, wq = torch.zeros(m, k).to(torch.float8_e4m3fn), torch.zeros(n, k).to(torch.float8_e4m3fn)
    xs, ws = torch.ones(m, 1), torch.ones(1, n)
    assert ops._e4m3_ok(q, xs, wq, ws, None)
    assert ops._e4m3_ok(q, xs, torch.nn.Parameter(wq, requires_grad=False), ws, torch.empty(m, n, dtype=torch.bfloat16))
    said = []

    def ask(q, xs):
        said.append(ops._e4m3_ok(q, xs, wq, ws, None))
        return xs * 2
    with FakeTensorMode(allow_non_fake_inputs=True) as mode:
        ask(mode.from_tensor(q), mode.from_tensor(xs))
    make_fx(ask)(q, xs)
    make_fx(ask, tracing_mode="symbolic")(q, xs)
    torch.jit.trace(ask, (q, xs), check_trace=False)
    torch.vmap(ask, in_dims=(None, 0))(q, xs.unsqueeze(0))
    assert said and not any(said)
    for bad in (q[:0], q[:, :128], q.t(), q[0], q.float(), q[::2, :]):
        assert not ops._e4m3_ok(bad, xs[:len(bad)], wq, ws, None)
    assert not ops._e4m3_ok(q, xs.t(), wq, ws, None) and not ops._e4m3_ok(q, xs, wq[:, :128], ws, None) and not ops._e4m3_ok(q, xs, wq, ws.double(), None)
