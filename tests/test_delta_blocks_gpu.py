"""The delta rule's block kernels (``csrc/kernels/gatemix.hip``) at the edges of their 64-token blocks and 16-wide tiles, against 64 bits."""
import types

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _step(lens, starts):
    n = np.asarray(lens)
    t = lambda a: torch.as_tensor(np.asarray(a, dtype=np.int32)).cuda()
    tiles = [(i, q) for i, m in enumerate(lens) for q in range(0, m, 64)]
    return types.SimpleNamespace(num_decode=0, num_prefill=len(n), num_seqs=len(n), positions=t(np.concatenate([s + np.arange(m) for s, m in zip(starts, lens)])),
                                 query_start_loc=t(np.concatenate([[0], np.cumsum(n)])), token_seq=t(np.repeat(np.arange(len(n)), n)),
                                 state_slots=t(np.arange(len(n))[::-1].copy()), counts=t([0, 0, len(tiles), len(n)]),
                                 prefill_tile_seq=t([a for a, _ in tiles]), prefill_tile_q0=t([b for _, b in tiles]), num_prefill_tiles=len(tiles))


# value columns around a tile; D around its tiles; z and v whose rows begin off 16 bytes (`off`)
@pytest.mark.parametrize("channel,H,G,D,Dv,off", [(True, 2, 1, 128, 128, 0), (True, 2, 2, 64, 15, 1), (True, 3, 1, 17, 33, 0), (True, 130, 2, 16, 16, 0), (True, 64, 1, 16, 31, 0),
                                                  (False, 2, 1, 128, 128, 0), (False, 2, 2, 48, 1, 1), (False, 130, 2, 33, 31, 0), (False, 1, 1, 256, 17, 0)])
def test_delta_blocks_against_64_bits(channel, H, G, D, Dv, off):
    """Chains of one, two and six blocks that end before, at and behind a block's last token, walked in the order of their lengths; one continues
    a state.  What a token adds to the fp32 state is rounded a few times per step of the chain: 2e-6 of the largest value over up to 330 tokens."""
    from dli_amd.ops import seqmix
    lens, starts = [63, 64, 65, 128, 2, 330], [0, 9, 0, 0, 0, 0]
    g = torch.Generator(device="cuda").manual_seed(D * 7 + Dv)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    T, S = sum(lens), len(lens)
    meta = _step(lens, starts)
    unit = lambda x: torch.nn.functional.normalize(x.view(T, G, D), dim=-1).view(T, G * D)
    q, k = unit(rnd(T, G * D)), unit(rnd(T, G * D))
    v, z = rnd(T, H * Dv + 4)[:, off:off + H * Dv], rnd(T, H * D + 8)[:, off:off + H * D]
    weight, rate, bias = torch.rand(T, H, generator=g, device="cuda"), torch.rand(H, generator=g, device="cuda") + 0.1, rnd(H * D)
    state = rnd(S, H, D, Dv) * 0.3
    A = state.double().clone()
    if channel:
        log = -rate.double()[None, :, None] * torch.nn.functional.softplus(z.double() + bias.double()).view(T, H, D)
        got = seqmix.channel_delta_scan(q, k, v, z, rate, bias, weight, state, meta, H, G, D, Dv)
    else:
        decay = -torch.exp(2.0 * rnd(T, H) - 2.0)
        log = decay.double()[:, :, None].expand(T, H, D)
        got, _ = seqmix.gated_scan(q, k, v, decay, weight, state, meta, H, G, D, Dv, delta=True)
    heads = lambda x: x.double().view(T, G, D).repeat_interleave(H // G, 1)
    qd, kd, vd = heads(q), heads(k), v.double().reshape(T, H, Dv)
    want, t = torch.empty(T, H, Dv, dtype=torch.float64, device="cuda"), 0
    for i, n in enumerate(lens):
        slot = int(meta.state_slots[i])
        M = A[slot] if starts[i] else torch.zeros_like(A[slot])
        for t in range(t, t + n):
            M = torch.exp(log[t])[:, :, None] * M
            u = weight[t].double()[:, None] * (vd[t] - (M * kd[t][:, :, None]).sum(1))
            M = M + kd[t][:, :, None] * u[:, None]
            want[t] = (M * qd[t][:, :, None]).sum(1)
        t += 1
        A[slot] = M
    assert (got.view(T, H, Dv).double() - want).abs().max() <= 2e-6 * want.abs().max().clamp_min(1.0)
    assert (state.double() - A).abs().max() <= 2e-6 * A.abs().max().clamp_min(1.0)


def _inputs(T, seqs, H, D, Dv, channel):
    g = torch.Generator(device="cuda").manual_seed(T + D)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    unit = lambda x: torch.nn.functional.normalize(x, dim=-1)
    x = dict(q=unit(rnd(T, D)), k=unit(rnd(T, D)), v=rnd(T, H * Dv), weight=torch.rand(T, H, generator=g, device="cuda"))
    if channel:
        x["z"] = rnd(T, H * D)
    else:
        x["decay"] = -0.3 * torch.rand(T, H, generator=g, device="cuda")
    return x, torch.zeros(seqs, H, D, Dv, device="cuda")


def _scan(x, state, meta, H, D, Dv):
    from dli_amd.ops import seqmix
    if "z" in x:
        rate, bias = torch.full((H,), 0.3, device="cuda"), torch.zeros(H * D, device="cuda")
        return seqmix.channel_delta_scan(x["q"], x["k"], x["v"], x["z"], rate, bias, x["weight"], state, meta, H, 1, D, Dv)
    return seqmix.gated_scan(x["q"], x["k"], x["v"], x["decay"], x["weight"], state, meta, H, 1, D, Dv, delta=True)[0]


@pytest.mark.parametrize("channel", [False, True])
def test_order_of_the_tile_list_changes_nothing(channel):
    """A step's list is sorted over its sequences.  Chunks of 1, 64, 65 and 130 blocks, then the second one without a state slot."""
    lens, H, D, Dv = [40, 4096, 4097, 8300], 1, 32, 16
    x, zeros = _inputs(sum(lens), len(lens), H, D, Dv, channel)
    meta = _step(lens, [0] * len(lens))
    state = zeros.clone()
    want = _scan(x, state, meta, H, D, Dv)
    ts, t0, n = meta.prefill_tile_seq, meta.prefill_tile_q0, meta.num_prefill_tiles
    for order in (np.arange(n)[::-1].copy(), np.random.default_rng(3).permutation(n)):
        o = torch.as_tensor(order, device="cuda")
        meta.prefill_tile_seq, meta.prefill_tile_q0 = ts[o].contiguous(), t0[o].contiguous()
        again = zeros.clone()
        assert torch.equal(_scan(x, again, meta, H, D, Dv), want) and torch.equal(again, state)
    slot = int(meta.state_slots[1])
    meta.state_slots[1] = -1
    again = zeros.clone()
    got = _scan(x, again, meta, H, D, Dv)
    assert torch.equal(got[:40], want[:40]) and torch.equal(got[40 + 4096:], want[40 + 4096:])
    state[slot] = 0.0
    assert torch.equal(again, state)


def test_workspace_holds_tiles_not_batch_rows():
    """400 single tokens in front of prompts of 130 and 70 tokens take no rows of the workspace: five tiles of 4 heads of 128 × 128, and the results."""
    H, D, single = 4, 128, 400
    lens, tiles = [1] * single + [130, 70], [(single, 0), (single + 1, 0), (single, 64), (single + 1, 64), (single, 128)]
    x, state = _inputs(sum(lens), len(lens), H, D, D, False)
    meta = _step(lens, [0] * len(lens))
    t = lambda a: torch.as_tensor(np.asarray(a, dtype=np.int32)).cuda()
    meta.prefill_tile_seq, meta.prefill_tile_q0, meta.num_prefill_tiles = t([a for a, _ in tiles]), t([b for _, b in tiles]), len(tiles)
    meta.counts = t([0, 0, len(tiles), len(lens)])
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    got = _scan(x, state, meta, H, D, D)
    took = torch.cuda.max_memory_allocated() - before
    assert took <= 4 * sum(lens) * H * D + len(tiles) * H * (160 << 10) + (1 << 20), took
    alone = _scan({k: v[single:].contiguous() for k, v in x.items()}, torch.zeros(2, H, D, D, device="cuda"), _step([130, 70], [0, 0]), H, D, D)
    assert torch.equal(got[single:], alone)
