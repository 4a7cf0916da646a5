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
