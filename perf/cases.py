"""Timed work of the serving stack: what one step of a served model asks of ``dli_amd.ops``, one decoder layer at a time.

A server on this framework runs, per layer and step: rotation + cache write + paged attention (decode rows, prompt chunks or both),
the projections of the feed-forward (dense, W8A8 or routed experts), and once per step the sampler; stacks with other mixers run
attention over token-major pages or a recurrence with matrix states instead.  Every case is one of these paths at the layer
sizes of the repository's presets (``llama3-8b``, ``llama3-70b``, its eighth ``llama3-70b-tp8shard``, ``mixtral-8x7b``) and of its
mixer benchmark (widths 2048 and 4096).  Steps without prompt tokens are replayed from a captured hipGraph, as the engine replays
its decode steps; steps with prompts are called eagerly.  The GEMM dispatch is the untuned one (``EngineConfig.tune_gemms = False``):
measuring it belongs to a server's start-up.

The number formats are those served in earnest: bf16, e4m3 caches with calibrated per-head scales, W8A8 projections; the recurrences
keep their states and sums in fp32 whatever the model's type.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from dli_amd import ops
from dli_amd.ops import seqmix
from dli_amd.ops.kv_layout import allocate_kv_cache
from dli_amd.ops.reference import build_cos_sin_cache

PAGE = 32                       # tokens per cache page
HD = 128                        # head size of the paged-KV families
THETA = 500000.0
TAPS = 4                        # filter length in front of the recurrences
BF16 = torch.bfloat16
F8 = torch.float8_e4m3fn


# ------------------------------------------------------------------------------------------------ cases
def listed():
    return [
        # one user streaming an answer: the latency of the smallest step
        dict(name="decode-attention-single", kind="attention", heads=32, kv_heads=8, fp8=False, decode=1, context=620, prompts=0, new=0, prefix=0),
        # a loaded replica between prompts: conversations of all ages side by side, bound by the cache bytes
        dict(name="decode-attention-ragged", kind="attention", heads=32, kv_heads=8, fp8=False, decode=160, context=2048, prompts=0, new=0, prefix=0),
        # a step filled with fresh prompts of unequal length
        dict(name="prefill-attention", kind="attention", heads=32, kv_heads=8, fp8=False, decode=0, context=0, prompts=5, new=1333, prefix=0),
        # the usual step under load with an e4m3 cache: decode rows beside prompt chunks that continue a context
        dict(name="mixed-attention-fp8", kind="attention", heads=32, kv_heads=8, fp8=True, decode=96, context=1500, prompts=2, new=1024, prefix=1024),
        # norm + gated feed-forward of a few streams: weight streaming
        dict(name="mlp-decode", kind="mlp", hidden=4096, ffn=14336, rows=5, w8a8=False),
        # the same for an ordinary decode batch, between the streaming and the compute-bound regime
        dict(name="mlp-batch", kind="mlp", hidden=4096, ffn=14336, rows=96, w8a8=False),
        # a prompt chunk on the fp8 matrix cores
        dict(name="mlp-prefill-fp8", kind="mlp", hidden=4096, ffn=14336, rows=2000, w8a8=True),
        # routed experts of a decode batch: every expert sees a handful of rows
        dict(name="moe-decode", kind="moe", hidden=4096, ffn=14336, experts=8, top_k=2, rows=40),
        # routed experts of a full prefill step
        dict(name="moe-prefill", kind="moe", hidden=4096, ffn=14336, experts=8, top_k=2, rows=4096),
        # the sampler of a decode batch whose requests ask for different things: greedy, plain draws, nucleus, top-k
        dict(name="sample-batch", kind="sample", vocab=128256, rows=57),
        # prompts through sliding-window attention with distance penalties over token-major pages
        dict(name="window-prefill", kind="tokens", mask="window", heads=32, kv_heads=8, decode=0, context=0, prompts=4, new=1200),
        # prompts through the delta rule with a decay per key channel
        dict(name="recurrence-prefill", kind="recurrence", form="channel", heads=16, decode=0, prompts=4, new=1200),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(("attention", "attention", "mlp", "moe", "sample", "tokens", "recurrence"))
    if kind == "mlp":
        hidden, ffn = rng.choice(((4096, 14336), (8192, 3584)))
        return dict(kind=kind, hidden=hidden, ffn=ffn, rows=_log(rng, 1, 4096), w8a8=rng.random() < 0.34)
    if kind == "moe":
        return dict(kind=kind, hidden=4096, ffn=14336, experts=8, top_k=2, rows=_log(rng, 1, 4096))
    if kind == "sample":
        return dict(kind=kind, vocab=rng.choice((32000, 128256)), rows=_log(rng, 1, 512))
    new = _log(rng, 17, 2048)
    prompts = rng.randint(1, max(1, min(16, 3600 // new)))
    what = rng.choice(("decode", "prefill", "mixed") if kind != "recurrence" else ("decode", "prefill"))
    decode = _log(rng, 1, 512 if kind == "attention" else 256) if what != "prefill" else 0
    context = _log(rng, 40, 2048) if what != "prefill" else 0
    if what == "decode":
        prompts = new = 0
    if kind == "attention":
        heads, kv_heads = rng.choice(((32, 8), (32, 8), (64, 8), (8, 1)))
        prefix = 0 if what == "decode" or rng.random() < 0.5 else rng.randint(1, 1500)
        return dict(kind=kind, heads=heads, kv_heads=kv_heads, fp8=rng.random() < 0.34, decode=decode, context=context, prompts=prompts,
                    new=new, prefix=prefix)
    if kind == "tokens":
        heads, kv_heads = rng.choice(((16, 4), (32, 8)))
        return dict(kind=kind, mask=rng.choice(("window", "chunk", "latent")), heads=heads, kv_heads=kv_heads, decode=decode, context=context,
                    prompts=prompts, new=new)
    return dict(kind=kind, form=rng.choice(("delta", "channel")), heads=rng.choice((16, 32)), decode=decode, prompts=prompts, new=new)


# ------------------------------------------------------------------------------------------------ a step's rows
def _spread(n, lo, hi):
    """``n`` unequal whole numbers from ``lo`` to ``hi`` (the last of them alone for one)."""
    if n == 1:
        return [hi]
    return [lo + int((hi - lo + 1) * ((i + 1) * 0.6180339887498949 % 1.0)) for i in range(n)]


def _rows(case):
    """(new tokens, context before them) of every sequence of the step: decode rows first."""
    nd, ctx = case["decode"], case.get("context", 0)
    ctx = ctx or 300                                              # a recurrence does not read its context
    rows = [(1, c) for c in (_spread(nd, max(ctx // 16, 1), ctx) if nd else [])]
    if case["prompts"]:
        new = _spread(case["prompts"], max(case["new"] // 4, 2), case["new"])
        pre = _spread(case["prompts"], 0, case.get("prefix", 0)) if case.get("prefix", 0) else [0] * len(new)
        rows += list(zip(new, pre))
    return rows


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape, scale=1.0, dtype=BF16):
    if dtype == BF16 and scale == 1.0:
        return torch.randn(*shape, generator=g, device="cuda", dtype=BF16)
    return (torch.randn(*shape, generator=g, device="cuda") * scale).to(dtype)


def _int32(a):
    return torch.from_numpy(np.ascontiguousarray(np.asarray(a, dtype=np.int32))).cuda()


class _Step:
    """Host-side layout of one step: pages in shuffled order, slots, positions, row offsets."""

    def __init__(self, case, seed):
        rows = _rows(case)
        self.nd, self.B = case["decode"], len(rows)
        self.new = np.array([n for n, _ in rows])
        self.ctx = np.array([c for _, c in rows])
        self.L = self.new + self.ctx
        self.T = int(self.new.sum())
        self.qsl = np.concatenate([[0], np.cumsum(self.new)])
        pages = (self.L + PAGE - 1) // PAGE
        self.num_pages = int(pages.sum()) + 1
        order = np.random.default_rng(seed).permutation(self.num_pages)
        self.bt = np.zeros((self.B, int(pages.max())), dtype=np.int64)
        first = 0
        for i, n in enumerate(pages):
            self.bt[i, :n] = order[first:first + n]
            first += int(n)
        self.pos = np.concatenate([c + np.arange(n) for n, c in rows])
        self.seq = np.repeat(np.arange(self.B), self.new)
        self.slot = self.bt[self.seq, self.pos // PAGE] * PAGE + self.pos % PAGE

    def slots_of(self, i, lo, hi):
        t = np.arange(lo, hi)
        return self.bt[i, t // PAGE] * PAGE + t % PAGE

    def meta(self, tile_tokens):
        ts, t0 = ops.build_prefill_tiles(self.new[self.nd:], self.nd, tile_tokens, self.L[self.nd:])
        return ops.AttnMetadata(num_decode=self.nd, num_prefill=self.B - self.nd, num_tokens=self.T, positions=_int32(self.pos),
                                slot_mapping=_int32(self.slot), block_tables=_int32(self.bt), seq_lens=_int32(self.L),
                                query_start_loc=_int32(self.qsl), max_seq_len=int(self.L.max()), counts=_int32([0, 0, len(ts), self.B]),
                                prefill_tile_seq=_int32(ts), prefill_tile_q0=_int32(t0), num_prefill_tiles=len(ts),
                                token_seq=_int32(self.seq), state_slots=_int32(np.arange(self.B)), num_seqs=self.B)


def _captured(call, keep=()):
    """``call`` captured into a hipGraph, as the engine captures a decode step; ``keep``: tensors the passes move on, put back.  The
    graph holds addresses only: the tensors that ``call`` names stay alive with the result."""
    saved = [t.clone() for t in keep]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            call()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side, capture_error_mode=ops.CAPTURE_MODE):
        out = call()
    for t, s in zip(keep, saved):
        t.copy_(s)

    def replay():
        graph.replay()
        return out
    return replay, call


# ------------------------------------------------------------------------------------------------ inputs
def _attention_inputs(case, seed):
    g = _gen(seed)
    st = _Step(case, seed)
    H, G = case["heads"], case["kv_heads"]
    qkv = _randn(g, st.T, (H + 2 * G) * HD)
    past = int(st.ctx.sum())
    old = _randn(g, past, 2 * G * HD)                             # keys and values of the contexts, sequence by sequence
    return st, qkv, old


def _token_inputs(case, seed):
    g = _gen(seed)
    st = _Step(case, seed)
    H, G = (case["heads"], 1) if case["mask"] == "latent" else (case["heads"], case["kv_heads"])
    x = {}
    if case["mask"] == "latent":
        x["q1"] = _randn(g, H, st.T, 512, scale=0.5)
        x["q2"] = _randn(g, st.T, H, 192)
        x["k"], x["v"] = _randn(g, st.num_pages, PAGE, 576), None
    else:
        x["q1"], x["q2"] = _randn(g, st.T, H, HD), None
        x["k"], x["v"] = _randn(g, st.num_pages, PAGE, G * HD), _randn(g, st.num_pages, PAGE, G * HD)
    f32 = dict(dtype=torch.float32)
    x["temp"] = 1.0 + _randn(g, H, scale=0.1, **f32)
    x["r1"], x["r2"] = (_randn(g, H, scale=0.1, **f32).abs() for _ in range(2))
    x["sink"] = _randn(g, H, **f32)
    return st, H, G, x


def _recurrence_inputs(case, seed):
    g = _gen(seed)
    st = _Step(case, seed)
    H = case["heads"]
    G, D = H // 2, HD
    C = (2 * G + H) * D
    cols = C + (H * D + 2 * H if case["form"] == "delta" else 256 + H)
    x = {"proj": _randn(g, st.T, (cols + 15) // 16 * 16), "taps": _randn(g, TAPS, C, scale=0.5, dtype=torch.float32)}
    x["low"] = _randn(g, st.T, 2 * H * D)
    x["rate"] = torch.exp(2.0 * torch.rand(H, generator=g, device="cuda"))
    x["bias"] = -4.0 + _randn(g, H if case["form"] == "delta" else H * D, dtype=torch.float32)
    x["norm"] = 1.0 + _randn(g, D, scale=0.1, dtype=torch.float32)
    x["state"] = _randn(g, st.B, H, D, D, scale=0.1, dtype=torch.float32)
    x["shift"] = _randn(g, st.B, TAPS - 1, C, dtype=torch.float32)
    return st, H, G, D, C, x


def _mlp_inputs(case, seed):
    g = _gen(seed)
    h, f = case["hidden"], case["ffn"]
    x = _randn(g, case["rows"], h, scale=2.0)
    norm = 1.0 + _randn(g, h, scale=0.1)
    return x, norm.to(BF16), _randn(g, 2 * f, h).mul_(h ** -0.5), _randn(g, h, f).mul_(f ** -0.5)


def _moe_inputs(case, seed):
    g = _gen(seed)
    h, f, e = case["hidden"], case["ffn"], case["experts"]
    return _randn(g, case["rows"], h), _randn(g, case["rows"], e), _randn(g, e, 2 * f, h).mul_(h ** -0.5), _randn(g, e, h, f).mul_(f ** -0.5)


def _kv_scales(old, new, G):
    """Calibrated e4m3 scales per head, 20 % head-room over what was seen (``ModelRunner.calibrate_kv_scales``)."""
    kv = torch.cat([old, new]).float().view(-1, 2, G, HD)
    k = kv[:, 0].view(-1, G, 2, HD // 2).pow(2).sum(2).sqrt().amax((0, 2))       # a pair's length bounds its rotations
    return torch.stack([k, kv[:, 1].abs().amax((0, 2))]) * (1.2 / 448.0)


def prepare(case, seed):
    kind = case["kind"]
    with torch.inference_mode():
        if kind == "attention":
            H, G = case["heads"], case["kv_heads"]
            st, qkv, old = _attention_inputs(case, seed)
            kc, vc = allocate_kv_cache(1, st.num_pages, G, HD, F8 if case["fp8"] else BF16, "cuda")[0]
            scales = _kv_scales(old, qkv[:, H * HD:], G) if case["fp8"] else None
            if old.shape[0]:                                      # the contexts, written by the steps before this one
                slots = np.concatenate([st.slots_of(i, 0, int(c)) for i, c in enumerate(st.ctx)])
                wide = torch.cat([old.new_zeros(old.shape[0], H * HD), old], dim=1)
                ops.rope_and_cache(wide, _int32(np.zeros(len(slots))), None, _int32(slots), kc, vc, H, G, HD, kv_scales=scales)
            meta = st.meta(ops.prefill_tile_tokens(H, G))
            if st.nd:
                ops.attach_decode_worklist(meta, st.L[:st.nd], H, G, "cuda")
            table = build_cos_sin_cache(8192, HD, THETA, "cuda")
            scale = HD ** -0.5

            def call():
                ops.rope_and_cache(qkv, meta.positions, table, meta.slot_mapping, kc, vc, H, G, HD, kv_scales=scales)
                return {"out": ops.paged_attention(qkv, kc, vc, meta, H, G, HD, scale, kv_scales=scales), "qkv": qkv}
            return _state(call, not case["prompts"], (qkv,))
        if kind == "mlp":
            x, norm, w13, w2 = _mlp_inputs(case, seed)
            if case["w8a8"]:
                (q13, s13), (q2, s2) = ops.quant_weight_fp8(w13), ops.quant_weight_fp8(w2)
                del w13, w2

                def call():
                    if case["rows"] < ops.FP8_MIN_ROWS:           # e4m3 weights streamed, activations kept in bf16
                        return ops.linear_w8(ops.linear_w8(ops.rms_norm(x, norm, 1e-5), q13, s13, swiglu=True), q2, s2)
                    gu = ops.linear_fp8(None, q13, s13, xq=ops.rms_norm_quant(x, None, norm, 1e-5))
                    return ops.linear_fp8(None, q2, s2, xq=ops.quant_rows_fp8(gu, silu=True))
            else:
                def call():
                    return ops.linear(ops.linear_swiglu(ops.rms_norm(x, norm, 1e-5), w13), w2)
            return _state(call, case["rows"] <= 256)
        if kind == "moe":
            x, logits, w13, w2 = _moe_inputs(case, seed)

            def call():
                return ops.fused_moe(x, logits, w13, w2, case["top_k"])
            return _state(call, case["rows"] <= 256)
        if kind == "sample":
            g = _gen(seed)
            B, V = case["rows"], case["vocab"]
            logits = torch.randn(B, V, generator=g, device="cuda") * 2.5
            likely = torch.randint(0, V, (B, 32), generator=g, device="cuda")
            logits.scatter_add_(1, likely, 12.0 * torch.rand(B, 32, generator=g, device="cuda"))
            logits = logits.to(BF16)
            i = np.arange(B)
            temp = torch.from_numpy(np.where(i % 4 == 0, 0.0, 0.7 + 0.1 * (i % 5)).astype(np.float32)).cuda()
            top_p = torch.from_numpy(np.where(i % 4 == 2, 0.9 + 0.01 * (i % 7), 1.0).astype(np.float32)).cuda()
            top_k = _int32(np.where(i % 4 == 3, 20 + i % 80, 0))
            seeds = torch.randint(0, 1 << 62, (B,), generator=g, device="cuda")
            steps = torch.randint(0, 1000, (B,), generator=g, device="cuda")
            return _state(lambda: ops.sample(logits, temp, top_p, top_k, seeds, steps), True)
        if kind == "tokens":
            st, H, G, x = _token_inputs(case, seed)
            meta = st.meta(seqmix.PREFILL_TILE_TOKENS)
            if case["mask"] == "latent":
                q1, q2 = x["q1"].transpose(0, 1), x["q2"][:, :, 128:]

                def call():
                    o = torch.empty(H, st.T, 512, dtype=BF16, device="cuda")
                    seqmix.token_attention(o.transpose(0, 1), q1, q2, x["k"], None, meta, 1, 512, 192 ** -0.5)
                    return o
            elif case["mask"] == "chunk":
                def call():
                    o = torch.empty(st.T, H, HD, dtype=BF16, device="cuda")
                    return seqmix.token_attention(o, x["q1"], None, x["k"], x["v"], meta, G, HD, HD ** -0.5, sink=x["sink"], chunk=1024)
            else:
                def call():
                    o = torch.empty(st.T, H, HD, dtype=BF16, device="cuda")
                    return seqmix.token_attention(o, x["q1"], None, x["k"], x["v"], meta, G, HD, HD ** -0.5, 1024, x["temp"], x["r1"], x["r2"])
            return _state(call, not case["prompts"])
        st, H, G, D, C, x = _recurrence_inputs(case, seed)
        meta = st.meta(seqmix.PREFILL_TILE_TOKENS)
        proj, state, shift = x["proj"], x["state"], x["shift"]
        unit = (2 * G, D, G, D ** -0.5)

        def call():
            out = torch.empty(st.T, H * D, dtype=BF16, device="cuda")
            if case["form"] == "delta":
                qkv, decay, beta = seqmix.causal_conv(proj[:, :C], x["taps"], None, shift, meta, torch.float32, act="silu", unit=unit,
                                                      gates=("delta", proj[:, C + H * D:C + H * D + 2 * H], x["rate"], x["bias"]))
                o, _ = seqmix.gated_scan(qkv[:, :G * D], qkv[:, G * D:2 * G * D], qkv[:, 2 * G * D:], decay, beta, state, meta, H, G, D, D,
                                         delta=True)
                seqmix.rms_gate(o, x["norm"], 1e-5, proj[:, C:C + H * D], BF16, groups=H, gate_act="silu", out=out, token_seq=meta.token_seq)
            else:
                qkv, _, beta = seqmix.causal_conv(proj[:, :C], x["taps"], None, shift, meta, torch.float32, act="silu", unit=unit,
                                                  gates=("beta", proj[:, C + 256:C + 256 + H], x["rate"], x["rate"]))
                o = seqmix.channel_delta_scan(qkv[:, :G * D], qkv[:, G * D:2 * G * D], qkv[:, 2 * G * D:], x["low"][:, :H * D], x["rate"],
                                              x["bias"], beta, state, meta, H, G, D, D)
                seqmix.rms_gate(o, x["norm"], 1e-5, x["low"][:, H * D:], BF16, groups=H, out=out, token_seq=meta.token_seq)
            return {"out": out, "state": state, "shift": shift}
        return _state(call, not case["prompts"], (state, shift))


def _state(call, captured, keep=()):
    one_pass, step = _captured(call, keep) if captured else (call, call)
    return {"pass": one_pass, "step": step}


def run(state):
    with torch.inference_mode():
        return state["pass"]()


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def work(case):
    kind = case["kind"]
    if kind == "mlp":
        m, h, f = case["rows"], case["hidden"], case["ffn"]
        return {"bytes": 3 * h * f * (1 if case["w8a8"] else 2) + 4 * m * h, "flops": 6 * m * h * f}
    if kind == "moe":
        m, h, f, e, k = case["rows"], case["hidden"], case["ffn"], case["experts"], case["top_k"]
        seen = e * (1.0 - (1.0 - k / e) ** m)                     # experts that get a row
        return {"bytes": 6 * seen * h * f + 4 * m * h + 2 * m * e, "flops": 6 * m * k * h * f}
    if kind == "sample":
        return {"bytes": case["rows"] * (2 * case["vocab"] + 36), "flops": 4 * case["rows"] * case["vocab"]}
    rows = _rows(case)
    T = sum(n for n, _ in rows)
    if kind == "attention":
        H, G, e = case["heads"], case["kv_heads"], 1 if case["fp8"] else 2
        pairs = sum(n * c + n * (n + 1) // 2 for n, c in rows)
        return {"bytes": 4 * T * (H + 2 * G) * HD + 2 * T * H * HD + sum(n + c for n, c in rows) * 2 * G * HD * e, "flops": 4 * H * HD * pairs}
    H = case["heads"]
    if kind == "tokens":
        reach = {"window": lambda p: min(p + 1, 1024), "chunk": lambda p: p % 1024 + 1, "latent": lambda p: p + 1}[case["mask"]]
        pairs = sum(reach(c + j) for n, c in rows for j in range(n))
        keys = sum(min(n + c, n - 1 + reach(c)) for n, c in rows)
        dk, dv, row = (576, 512, 576) if case["mask"] == "latent" else (HD, HD, 2 * case["kv_heads"] * HD)
        return {"bytes": 2 * T * H * (dk + dv) + 2 * keys * row, "flops": 2 * H * (dk + dv) * pairs}
    D, G = HD, H // 2
    C = (2 * G + H) * D
    gates = H * D + 2 * H if case["form"] == "delta" else 2 * H * D + H
    kept = len(rows) * (H * D * D + (TAPS - 1) * C) * 4
    return {"bytes": 2 * T * (C + gates + H * D) + kept * (2 if case["decode"] else 1), "flops": 6 * T * H * D * D}


# ------------------------------------------------------------------------------------------------ how exact
def tolerance(case):
    """About four times what was measured against 64 bits with bf16 operands and results: 0.0027 for paged attention (0.0076 with an e4m3
    cache), 0.0042 for two products in a row (0.046 with e4m3 activations: more than a comparison may allow), 0.003 for routed experts,
    0.0017 behind fp32 sums."""
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind == "attention":
        return {"rel": 0.03, "max": 0.5} if case["fp8"] else {"rel": 0.011, "max": 0.25}
    if kind == "mlp":
        return {"rel": 0.03, "max": 0.6} if case["w8a8"] else {"rel": 0.017, "max": 0.25}
    if kind == "moe":
        return {"rel": 0.012, "max": 0.25}
    return {"rel": 0.007, "max": 0.1}


def _softmax_attend(q, k, v, bias):
    s = torch.softmax(q @ k.transpose(-1, -2) + bias, dim=-1)
    return s @ v


def _exact_attention(case, seed):
    H, G = case["heads"], case["kv_heads"]
    st, qkv, old = _attention_inputs(case, seed)
    scales = _kv_scales(old, qkv[:, H * HD:], G).double() if case["fp8"] else None
    x = qkv.double().view(st.T, H + 2 * G, HD)
    pos = torch.from_numpy(st.pos).cuda()
    ang = pos.double()[:, None] * (THETA ** (-torch.arange(0, HD, 2, dtype=torch.float64, device="cuda") / HD))[None]
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x[:, :H + G, :HD // 2], x[:, :H + G, HD // 2:]
    x = torch.cat([torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1), x[:, H + G:]], dim=1)

    def stored(t, which):                                         # what the cache keeps of context keys / values
        if scales is None:
            return t
        s = scales[which][None, :, None]
        return (t.float() / s.float()).clamp(-448, 448).to(F8).double() * s
    out = torch.empty(st.T, H, HD, dtype=torch.float64, device="cuda")
    first = np.concatenate([[0], np.cumsum(st.ctx)])
    for i in range(st.B):
        o = old[first[i]:first[i + 1]].double().view(-1, 2, G, HD)
        t0, t1 = int(st.qsl[i]), int(st.qsl[i + 1])
        k = torch.cat([stored(o[:, 0], 0), stored(x[t0:t1, H:H + G], 0)])
        v = torch.cat([stored(o[:, 1], 1), stored(x[t0:t1, H + G:], 1)])
        n, L = t1 - t0, int(st.L[i])
        far = torch.arange(L, device="cuda")[None] > (L - n + torch.arange(n, device="cuda"))[:, None]
        bias = torch.zeros(n, L, dtype=torch.float64, device="cuda").masked_fill_(far, -torch.inf)
        for h in range(G):
            q = x[t0:t1, h * (H // G):(h + 1) * (H // G)].transpose(0, 1) * HD ** -0.5
            out[t0:t1, h * (H // G):(h + 1) * (H // G)] = _softmax_attend(q, k[:, h], v[:, h], bias).transpose(0, 1)
    return {"out": out.reshape(st.T, -1), "qkv": x.reshape(st.T, -1)}


def _exact_tokens(case, seed):
    st, H, G, x = _token_inputs(case, seed)
    latent = case["mask"] == "latent"
    dv = 512 if latent else HD
    out = torch.empty(st.T, H, dv, dtype=torch.float64, device="cuda")
    for i in range(st.B):
        t0, t1, L = int(st.qsl[i]), int(st.qsl[i + 1]), int(st.L[i])
        slots = torch.from_numpy(st.slots_of(i, 0, L)).cuda()
        k = x["k"].view(-1, x["k"].shape[-1])[slots].double().view(L, G, -1)
        v = k[:, :, :512] if latent else x["v"].view(-1, G * HD)[slots].double().view(L, G, HD)
        p = torch.arange(L - (t1 - t0), L, device="cuda")[:, None]
        j = torch.arange(L, device="cuda")[None]
        hidden = j > p
        if case["mask"] == "window":
            hidden = hidden | (p - j >= 1024)
        if case["mask"] == "chunk":
            hidden = hidden | (j < p - p % 1024)
        for h in range(H):
            q = (torch.cat([x["q1"][h, t0:t1], x["q2"][t0:t1, h, 128:]], dim=1) if latent else x["q1"][t0:t1, h]).double()
            s = q @ k[:, h // (H // G)].t() * (192 ** -0.5 if latent else HD ** -0.5)
            if case["mask"] == "window":
                s = s * x["temp"][h].double() - x["r1"][h].double() * torch.log1p(x["r2"][h].double() * (p - j).clamp(min=0))
            s = s.masked_fill(hidden, -torch.inf)
            if case["mask"] == "chunk":
                s = torch.cat([s, x["sink"][h].double().expand(t1 - t0, 1)], dim=1)
            out[t0:t1, h] = torch.softmax(s, dim=1)[:, :L] @ v[:, h // (H // G)]
    return out.transpose(0, 1).contiguous() if latent else out


def _exact_recurrence(case, seed):
    st, H, G, D, C, x = _recurrence_inputs(case, seed)
    proj = x["proj"].double()
    n = int(st.new.max())
    new, fresh = torch.from_numpy(st.new).cuda(), torch.from_numpy(st.ctx == 0).cuda()
    rows = torch.from_numpy(st.seq).cuda(), torch.from_numpy(st.pos - st.ctx[st.seq]).cuda()

    def padded(t, width):                                         # [T, …] → [B, n, …]
        p = t.new_zeros(st.B, n, width)
        p[rows] = t
        return p
    hist = torch.where(fresh[:, None, None], 0.0, x["shift"].double())
    ext = torch.cat([hist, padded(proj[:, :C], C)], dim=1)
    conv = sum(x["taps"][j].double() * ext[:, j:j + n] for j in range(TAPS))
    conv = torch.nn.functional.silu(conv)
    shift = torch.stack([ext[i, int(new[i]):int(new[i]) + TAPS - 1] for i in range(st.B)])
    del ext, hist
    qk = conv[:, :, :2 * G * D].view(st.B, n, 2 * G, D)
    qk = qk * torch.rsqrt((qk * qk).sum(-1, keepdim=True) + 1e-6)
    q = (qk[:, :, :G] * D ** -0.5).repeat_interleave(H // G, dim=2)
    k = qk[:, :, G:].repeat_interleave(H // G, dim=2)
    v = conv[:, :, 2 * G * D:].view(st.B, n, H, D)
    if case["form"] == "delta":
        gate, b = proj[:, C:C + H * D], proj[:, C + H * D:]
        beta = padded(torch.sigmoid(b[:, :H]), H)
        g = torch.exp(-x["rate"].double() * torch.nn.functional.softplus(b[:, H:2 * H] + x["bias"].double()))
        g = padded(g, H)[:, :, :, None]
        act = torch.nn.functional.silu(gate)
    else:
        low = x["low"].double()
        beta = padded(torch.sigmoid(proj[:, C + 256:C + 256 + H]), H)
        z = torch.nn.functional.softplus(low[:, :H * D] + x["bias"].double()).view(-1, H, D)
        g = padded(torch.exp(-x["rate"].double()[None, :, None] * z).reshape(-1, H * D), H * D).view(st.B, n, H, D)
        act = torch.sigmoid(low[:, H * D:])
    S = torch.where(fresh[:, None, None, None], 0.0, x["state"].double())
    o = S.new_zeros(st.B, n, H, D)
    for t in range(n):
        on = (new > t)[:, None, None, None]
        A = g[:, t, :, :, None] * S
        u = beta[:, t, :, None] * (v[:, t] - torch.matmul(k[:, t, :, None, :], A)[:, :, 0])
        A = A + k[:, t, :, :, None] * u[:, :, None, :]
        o[:, t] = torch.matmul(q[:, t, :, None, :], A)[:, :, 0]
        S = torch.where(on, A, S)
    o = o[rows]
    o = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + 1e-5) * x["norm"].double()
    return {"out": o.view(st.T, H * D) * act, "state": S, "shift": shift}


def exact(case, seed):
    kind = case["kind"]
    with torch.inference_mode():
        if kind == "attention":
            return _exact_attention(case, seed)
        if kind == "tokens":
            return _exact_tokens(case, seed)
        if kind == "recurrence":
            return _exact_recurrence(case, seed)
        if kind == "mlp":
            x, norm, w13, w2 = _mlp_inputs(case, seed)
            x = x.double()
            x = x * torch.rsqrt((x * x).mean(1, keepdim=True) + 1e-5) * norm.double()
            if case["w8a8"]:                                      # the weights are e4m3 from the start
                def kept(w):
                    s = w.float().abs().amax(dim=1, keepdim=True).clamp_min(1e-12) / 448.0
                    return (w.float() / s).clamp(-448, 448).to(F8).double() * s.double()
                w13, w2 = kept(w13), kept(w2)
            y = x @ w13.double().t()
            y = torch.nn.functional.silu(y[:, :case["ffn"]]) * y[:, case["ffn"]:]
            return y @ w2.double().t()
        if kind == "moe":
            x, logits, w13, w2 = _moe_inputs(case, seed)
            p = logits.double()
            ids = torch.sort(p, dim=1, descending=True, stable=True).indices[:, :case["top_k"]]
            wts = torch.softmax(torch.gather(p, 1, ids), dim=1)
            out = torch.zeros(case["rows"], case["hidden"], dtype=torch.float64, device="cuda")
            for e in range(case["experts"]):
                t, s = torch.nonzero(ids == e, as_tuple=True)
                if len(t):
                    y = x[t].double() @ w13[e].double().t()
                    y = torch.nn.functional.silu(y[:, :case["ffn"]]) * y[:, case["ffn"]:]
                    out.index_add_(0, t, (y @ w2[e].double().t()) * wts[t, s, None])
            return out
        return None                                               # token ids: whole numbers, compared as they are
