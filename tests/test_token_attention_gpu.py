"""Decode rows over token-major pages: whole and split key ranges, page remainders, one row as key and value, shared heads."""
import pytest
import torch

from dli_amd.ops import AttnMetadata, seqmix

pytestmark = pytest.mark.gpu
PAGE = 32
_INF = float("inf")


def _rows(lens, seed):
    """Pages of the rows in a shuffled order; the last row is padding."""
    n = [-(-x // PAGE) for x in lens]
    order = (torch.randperm(sum(n), generator=torch.Generator().manual_seed(seed)) + 1).int()
    tables = torch.zeros(len(lens) + 1, max(n), dtype=torch.int32)
    at = 0
    for i, k in enumerate(n):
        tables[i, :k] = order[at:at + k]
        at += k
    return tables, sum(n) + 1


def _exact(q, k, v, tables, lens, G, scale, window, cap):
    out = torch.zeros(len(lens) + 1, q.shape[1], v.shape[-1], dtype=torch.float64)
    per = q.shape[1] // G
    for i, x in enumerate(lens):
        j = torch.arange(max(0, x - window) if window else 0, x)
        at = tables[i, j // PAGE].long() * PAGE + j % PAGE
        for h in range(q.shape[1]):
            s = k[at, h // per].double() @ q[i, h].double() * scale
            s = cap * torch.tanh(s / cap) if cap else s
            out[i, h] = torch.softmax(s, 0) @ v[at, h // per].double()
    return out


@pytest.mark.parametrize("lens", [[1], [31, 32, 33, 65], [700], [257] * 70])
@pytest.mark.parametrize("H,G,Dk,Dv,shared", [(8, 1, 24, 16, False), (16, 2, 128, 128, False), (20, 1, 72, 80, False), (32, 1, 576, 512, True),
                                              (8, 1, 320, 512, False), (24, 2, 192, 64, True), (6, 2, 20, 33, False),
                                              (32, 8, 128, 128, False), (14, 2, 200, 176, False), (10, 2, 8, 16, False), (4, 1, 96, 96, True)])
def test_decode_rows(H, G, Dk, Dv, shared, lens):
    g = torch.Generator().manual_seed(H * Dk + len(lens))
    tables, pages = _rows(lens, Dk)
    T = len(lens) + 1
    q = torch.randn(T, H, Dk, generator=g).bfloat16()
    k = torch.randn(pages * PAGE, G, Dk, generator=g).bfloat16()
    v = k[..., :Dv] if shared else torch.randn(pages * PAGE, G, Dv, generator=g).bfloat16()
    scale = Dk ** -0.5
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    meta = AttnMetadata(num_decode=T, num_prefill=0, num_tokens=T, positions=ints([x - 1 for x in lens] + [0]), slot_mapping=ints([-1] * T),
                        block_tables=tables.cuda(), seq_lens=ints(lens + [0]), query_start_loc=ints(range(T + 1)), token_seq=ints([*range(T - 1), -1]))
    for window, cap in ((0, 0.0), (40, 5.0)):
        want = _exact(q, k, v, tables, lens, G, scale, window, cap)
        for dtype in (torch.bfloat16, torch.float32):
            out = torch.full((T, H, Dv), float("nan"), dtype=dtype, device="cuda")
            seqmix.token_attention(out, q.cuda(), None, k.cuda().view(pages, PAGE, -1), None if shared else v.cuda().view(pages, PAGE, -1), meta, G, Dv,
                                   scale, window, cap=cap)
            got = out.double().cpu()
            # weights of 16 bits at least and scores to some 2^-20, times the largest value; bf16 results are rounded once more
            bound = float(v.abs().max()) * 2.0 ** -15 + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0.0)
            assert ((got - want).abs() <= bound).all(), (window, cap, dtype, (got - want).abs().max())
            assert not got[-1].any()


@pytest.mark.parametrize("options", ["window penalties", "steep penalties", "chunk sink", "gate kept"])
@pytest.mark.parametrize("H,G,D,rows", [(4, 1, 48, 1), (4, 1, 16, 1), (12, 2, 128, 70), (20, 4, 208, 3)])
def test_small_groups_as_a_lane_per_key_does(H, G, D, rows, options, monkeypatch):
    """Groups of 4 to 7 heads on the matrix cores against the kernel that takes a lane per key, whose weights are fp32 values."""
    g = torch.Generator().manual_seed(H + D)
    lens = [(37 * i + 260) % 300 + 1 for i in range(rows)]     # (one row: several pages, most slices empty)
    tables, pages = _rows(lens, D)
    rand = lambda *s: torch.randn(*s, generator=g).bfloat16().cuda()
    q, k, v = rand(rows, H, 2 * D)[..., D:], rand(pages, PAGE, G * D), rand(pages, PAGE, G * D)      # (queries with gaps between them)
    pos = lambda: torch.rand(H, generator=g).cuda()
    kw = {"window penalties": dict(window=50, temp=pos() + 0.5, r1=pos(), r2=pos()), "steep penalties": dict(r1=1e6 * (pos() + 0.5), r2=1e-6 * (pos() + 0.5)),   # (1 + r2 · distance has lost them)
          "chunk sink": dict(chunk=64, sink=pos()),
          "gate kept": dict(window=33, keep_first=40, gate=rand(rows, 3 * H)[:, H:2 * H], out_scale=1.5)}[options]
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    meta = AttnMetadata(num_decode=rows, num_prefill=0, num_tokens=rows, positions=ints([x - 1 for x in lens]), slot_mapping=ints([-1] * rows),
                        block_tables=tables.cuda(), seq_lens=ints(lens), query_start_loc=ints(range(rows + 1)), token_seq=ints(range(rows)))
    got, taken, lib = [], [], seqmix._hip()
    class Watched:
        def __getattr__(self, name):
            f = getattr(lib, name)
            return (lambda *a: taken.append(f(*a)) or taken[-1]) if name == "sm_head_decode_attention" else f
    monkeypatch.setattr(seqmix, "_hip", Watched)
    for on in (True, False):
        monkeypatch.setattr(seqmix, "HEAD_DECODE", on)
        out = torch.empty(H, rows, D, dtype=torch.bfloat16, device="cuda").transpose(0, 1)
        seqmix.token_attention(out, q, None, k, v, meta, G, D, D ** -0.5, **kw)
        got.append(out.float())
    assert taken == [True]                                     # the matrix cores took the first call
    # each result is rounded to bf16 from fp32 sums that differ by some 2^-20 of the largest value: one step apart at most
    assert ((got[0] - got[1]).abs() <= 2.0 ** -7 * got[1].abs() + 2.0 ** -18 * float(v.abs().max()) * 1.5).all()
    assert (got[0] != got[1]).float().mean() < 0.02


@pytest.mark.parametrize("options", [dict(), dict(window=40), dict(chunk=48), dict(window=40, keep_first=37)])
@pytest.mark.parametrize("H,G,Dk,Dv,shared", [(8, 2, 128, 128, False), (14, 2, 200, 176, False), (5, 1, 96, 96, True), (8, 1, 64, 64, False),
                                              (32, 1, 576, 512, True), (8, 1, 320, 512, False), (4, 2, 64, 64, False)])
def test_slots_that_a_row_does_not_see(H, G, Dk, Dv, shared, options):
    """Infinities and NaN past a row's position, before its window or chunk, and in its pages' other slots change nothing."""
    g = torch.Generator().manual_seed(Dk + H)
    lens = [1, 31, 33, 64, 100, 257]
    tables, pages = _rows(lens, Dk)
    T = len(lens)
    q = torch.randn(T, H, Dk, generator=g).bfloat16().cuda()
    k = torch.randn(pages, PAGE, G, Dk, generator=g).bfloat16()
    v = k[..., :Dv] if shared else torch.randn(pages, PAGE, G, Dv, generator=g).bfloat16()
    seen = torch.zeros(pages, PAGE, dtype=torch.bool)
    for i, x in enumerate(lens):
        p = x - 1
        low = max(0, p - options["window"] + 1) if "window" in options else p - p % options["chunk"] if "chunk" in options else 0
        for j in [*range(min(options.get("keep_first", 0), low)), *range(low, x)]:
            seen[tables[i, j // PAGE], j % PAGE] = True
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    meta = AttnMetadata(num_decode=T, num_prefill=0, num_tokens=T, positions=ints([x - 1 for x in lens]), slot_mapping=ints([-1] * T),
                        block_tables=tables[:T].cuda(), seq_lens=ints(lens), query_start_loc=ints(range(T + 1)), token_seq=ints(range(T)))
    out = []
    for other in (0.0, _INF, -_INF, float("nan")):
        k2, v2 = (torch.where(seen[..., None, None], x, torch.full_like(x, other)).cuda() for x in (k, v))
        out.append(torch.empty(T, H, Dv, dtype=torch.bfloat16, device="cuda"))
        seqmix.token_attention(out[-1], q, None, k2.view(pages, PAGE, -1), None if shared else v2.view(pages, PAGE, -1), meta, G, Dv, Dk ** -0.5, **options)
    assert bool(torch.isfinite(out[0].float()).all()) and all(torch.equal(o, out[0]) for o in out[1:])


@pytest.mark.parametrize("H,G,D", [(8, 2, 128), (14, 2, 208), (5, 1, 96)])
def test_infinite_values_that_small_groups_see(H, G, D, monkeypatch):
    """An infinite value is infinite in every head that sees it, as with the weights in fp32, and only there."""
    g = torch.Generator().manual_seed(D)
    lens = [1, 20, 33, 200]
    tables, pages = _rows(lens, D)
    T = len(lens)
    rand = lambda *s: torch.randn(*s, generator=g).bfloat16()
    q, k, v = rand(T, H, D).cuda(), rand(pages, PAGE, G * D).cuda(), rand(pages, PAGE, G * D)
    finite = v.clone()
    for i, x in enumerate(lens):                               # the last token of a row and its first: columns 3 and 16
        v[tables[i, (x - 1) // PAGE], (x - 1) % PAGE, 3::D] = _INF
        v[tables[i, 0], 0, 16::D] = -_INF
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    meta = AttnMetadata(num_decode=T, num_prefill=0, num_tokens=T, positions=ints([x - 1 for x in lens]), slot_mapping=ints([-1] * T),
                        block_tables=tables[:T].cuda(), seq_lens=ints(lens), query_start_loc=ints(range(T + 1)), token_seq=ints(range(T)))
    def run(values, on):
        monkeypatch.setattr(seqmix, "HEAD_DECODE", on)
        out = torch.empty(T, H, D, dtype=torch.bfloat16, device="cuda")
        return seqmix.token_attention(out, q, None, k, values.cuda(), meta, G, D, D ** -0.5).float()
    want = run(finite, True)
    want[..., 3], want[..., 16] = _INF, -_INF
    assert torch.equal(run(v, True), want)
    assert torch.equal(run(v, False).isinf(), want.isinf())    # (a lane per key)


@pytest.mark.parametrize("H,G,D", [(16, 2, 128), (8, 2, 128), (8, 1, 320)])
def test_slices_chosen_for_another_length(H, G, D):
    """The host's longest context chooses slices only: a step captured for short rows and replayed with longer ones is right too."""
    g = torch.Generator().manual_seed(D)
    lens = [40 + 13 * i for i in range(70)]
    tables, pages = _rows(lens, D)
    T = len(lens)
    rand = lambda *s: torch.randn(*s, generator=g).bfloat16()
    q, k, v = rand(T, H, D), rand(pages * PAGE, G, D), rand(pages * PAGE, G, D)
    want = _exact(q, k, v, tables, lens, G, D ** -0.5, 0, 0.0)[:T]
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    bound = float(v.abs().max()) * 2.0 ** -15 + 2.0 ** -8 * want.abs()     # as in test_decode_rows
    for longest in (0, 1, 300, max(lens)):
        meta = AttnMetadata(num_decode=T, num_prefill=0, num_tokens=T, positions=ints([x - 1 for x in lens]), slot_mapping=ints([-1] * T), max_seq_len=longest,
                            block_tables=tables[:T].cuda(), seq_lens=ints(lens), query_start_loc=ints(range(T + 1)), token_seq=ints(range(T)))
        out = torch.empty(T, H, D, dtype=torch.bfloat16, device="cuda")
        seqmix.token_attention(out, q.cuda(), None, k.cuda().view(pages, PAGE, -1), v.cuda().view(pages, PAGE, -1), meta, G, D, D ** -0.5)
        assert ((out.double().cpu() - want).abs() <= bound).all(), longest


def test_penalties_past_the_usual_range(monkeypatch):
    """r2 · distance of 0 to 1e38, and an r2 that is NaN, which makes its head NaN: on the matrix cores as with a lane per key."""
    g = torch.Generator().manual_seed(3)
    H, G, D, lens = 8, 2, 64, [1, 40, 200]
    tables, pages = _rows(lens, 5)
    T = len(lens)
    rand = lambda *s: torch.randn(*s, generator=g).bfloat16().cuda()
    q, k, v = rand(T, H, D), rand(pages, PAGE, G * D), rand(pages, PAGE, G * D)
    r1 = torch.full((H,), 2.0, device="cuda")
    r2 = torch.tensor([5e35, 1e30, 0.0, float("nan"), 1e-30, 1.0, 2.0 ** 24, 2.0 ** 17], device="cuda")
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    meta = AttnMetadata(num_decode=T, num_prefill=0, num_tokens=T, positions=ints([x - 1 for x in lens]), slot_mapping=ints([-1] * T),
                        block_tables=tables[:T].cuda(), seq_lens=ints(lens), query_start_loc=ints(range(T + 1)), token_seq=ints(range(T)))
    got = []
    for on in (True, False):
        monkeypatch.setattr(seqmix, "HEAD_DECODE", on)
        out = torch.empty(T, H, D, dtype=torch.bfloat16, device="cuda")
        got.append(seqmix.token_attention(out, q, None, k, v, meta, G, D, D ** -0.5, r1=r1, r2=r2).float())
    assert torch.equal(got[0].isnan(), got[1].isnan()) and got[0][:, 3].isnan().all() and got[0][:, 4:].isfinite().all()
    # one bf16 step, as in test_small_groups_as_a_lane_per_key_does
    assert torch.allclose(got[0], got[1], rtol=2.0 ** -7, atol=2.0 ** -18 * float(v.abs().max()) * 1.5, equal_nan=True)
