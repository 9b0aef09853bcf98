"""Timed workloads of the serving engine.

Every case is work that a serving step does, called the way the engine calls
it, at the layer widths of the named architectures:

  decode_step    one captured decode step of a Llama stack (graph replay)
  mixed_step     one eager step of a Llama stack: prompt portions beside the
                 single tokens of running conversations
  general_delta  the recurrence of a delta-rule mixer (ops.delta_rule)
  channel_delta  the recurrence with a decay per key channel (ops.gated_delta)
  scan           gated linear recurrences (ops.linear_scan: gla, ssd, mlstm)
  attention      paged attention with score mixing over heads, aligned chunks,
                 windows, kept first keys, capped scores, sinks
                 (ops.talk_attention)
  experts        a routed feed-forward of a decode batch, router to weighted
                 sum (ops.moe_route ... ops.experts_sum)

A case is a dict of plain values. Prompt lengths are ragged and follow from
the case alone; values follow from the seed. Weights and activations have the
distributions of the engine's own random initialisation.
"""

from __future__ import annotations

import dataclasses
import math
import random

import numpy as np
import torch

BLOCK = 16          # positions per cache page
EPS = 1e-5

_DT = {"bf16": torch.bfloat16, "f32": torch.float32}


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one conversation on the smallest chat model: launches and latency
        dict(name="decode_one", kind="decode_step", arch="llama-3.2-1b",
             layers=8, seqs=1, ctx_lo=517, ctx_hi=517, kv="auto"),
        # an ordinary decode batch; contexts from fresh to half a window
        dict(name="decode_batch", kind="decode_step", arch="llama-3-8b",
             layers=6, seqs=61, ctx_lo=300, ctx_hi=4000, kv="auto"),
        # a large decode batch on the fp8 key/value cache
        dict(name="decode_fp8_kv", kind="decode_step", arch="llama-3-8b",
             layers=4, seqs=192, ctx_lo=1200, ctx_hi=5500, kv="fp8"),
        # the multi-round question answering step: 320 users, a 2048-token
        # budget, histories of thousands of tokens
        dict(name="mixed_step", kind="mixed_step", arch="llama-3-8b",
             layers=4, seqs=313, ctx_lo=3600, ctx_hi=5600, prompts=4,
             tokens=1735, past=3700, kv="auto"),
        # prompt portions through the delta-rule layers of an 8b-sized stack
        dict(name="general_delta_prompt", kind="general_delta", heads=32,
             dim=128, prompts=2, tokens=8011, singles=0, past=4096,
             dtype="bf16"),
        # their decode batch: state in, state out
        dict(name="general_delta_decode", kind="general_delta", heads=32,
             dim=128, prompts=0, tokens=0, singles=64, past=1024,
             dtype="bf16"),
        # a step that mixes prompts and single tokens, grouped keys
        dict(name="channel_delta_mixed", kind="channel_delta", heads=32,
             kv_heads=16, dim=128, vdim=128, prompts=3, tokens=6007,
             singles=37, past=777, dtype="bf16"),
        # state-space heads of an 8b-sized stack
        dict(name="scan_ssd_prompt", kind="scan", mode="ssd", heads=128,
             groups=1, dim=128, vdim=64, prompts=2, tokens=8192, singles=0,
             past=0, dtype="bf16"),
        # gated linear attention at 1b width, one short prompt
        dict(name="scan_gla_prompt", kind="scan", mode="gla", heads=8,
             groups=8, dim=128, vdim=256, prompts=1, tokens=1501, singles=0,
             past=0, dtype="bf16"),
        # prompts through attention whose scores mix over the heads
        dict(name="talk_prompt", kind="attention", heads=32, kv_heads=8,
             dim=128, vdim=128, talk=True, chunk=2048, window=0,
             keep_first=0, softcap=0.0, prompts=2, tokens=4099, singles=0,
             past=0, ctx=0, dtype="bf16"),
        # windowed attention: prompts with history beside a decode batch
        dict(name="window_mixed", kind="attention", heads=32, kv_heads=8,
             dim=128, vdim=128, talk=False, chunk=0, window=2048,
             keep_first=4, softcap=30.0, prompts=2, tokens=8130, singles=61,
             past=1500, ctx=1800, dtype="bf16"),
        # routed feed-forward of a decode batch
        dict(name="experts_decode", kind="experts", width=4096, ff=3584,
             experts=8, top=2, rows=64, act="silu", score="softmax"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode_step", "mixed_step", "general_delta",
                       "channel_delta", "scan", "scan", "attention",
                       "attention", "experts"])
    if kind == "decode_step":
        arch = rng.choice(["llama-3.2-1b", "llama-3-8b"])
        lo = _log(rng, 40, 3000)
        return dict(kind=kind, arch=arch, layers=rng.choice([4, 5, 6]),
                    seqs=_log(rng, 1, 200), ctx_lo=lo,
                    ctx_hi=lo + _log(rng, 1, 2500),
                    kv=rng.choice(["auto", "auto", "fp8"]))
    if kind == "mixed_step":
        lo = _log(rng, 200, 3500)
        return dict(kind=kind, arch="llama-3-8b", layers=rng.choice([2, 3]),
                    seqs=_log(rng, 2, 300), ctx_lo=lo,
                    ctx_hi=lo + _log(rng, 10, 2000),
                    prompts=rng.randint(1, 6), tokens=_log(rng, 120, 1800),
                    past=rng.choice([0, _log(rng, 16, 4000)]),
                    kv=rng.choice(["auto", "auto", "fp8"]))
    if kind == "experts":
        return dict(kind=kind, width=rng.choice([2048, 4096]),
                    ff=rng.choice([2048, 3584, 1536]),
                    experts=rng.choice([8, 8, 16]), top=rng.choice([1, 2]),
                    rows=_log(rng, 1, 128),
                    act=rng.choice(["silu", "clamped_swish"]),
                    score=rng.choice(["softmax", "sigmoid"]))
    # prompts only, single tokens only, or both
    mix = rng.choice(["prompt", "prompt", "decode", "both"])
    ragged = dict(
        prompts=0 if mix == "decode" else rng.randint(1, 4),
        tokens=0 if mix == "decode" else _log(rng, 70, 6000),
        singles=0 if mix == "prompt" else _log(rng, 1, 128),
        past=rng.choice([0, _log(rng, 1, 3000)]),
        dtype=rng.choice(["bf16", "bf16", "bf16", "f32"]))
    if kind == "general_delta":
        dim = rng.choice([64, 128, 96])
        return dict(kind=kind, heads=rng.choice([8, 12, 32]), dim=dim,
                    **ragged)
    if kind == "channel_delta":
        kv = rng.choice([4, 8, 16])
        return dict(kind=kind, heads=kv * rng.choice([1, 2]), kv_heads=kv,
                    dim=rng.choice([64, 128, 96]),
                    vdim=rng.choice([64, 128, 80]), **ragged)
    if kind == "scan":
        mode = rng.choice(["gla", "ssd", "mlstm"])
        if mode == "gla":
            heads, dim, vdim = rng.choice([8, 16]), 128, 256
        elif mode == "ssd":
            heads, dim, vdim = rng.choice([48, 64, 128]), 128, 64
        else:
            heads, dim, vdim = rng.choice([16, 32]), 128, 128
        groups = rng.choice([1, heads // 8]) if mode == "ssd" else heads
        return dict(kind=kind, mode=mode, heads=heads, groups=groups,
                    dim=dim, vdim=vdim, **ragged)
    talk = rng.choice([True, False])
    dim = rng.choice([64, 128])
    limit = rng.choice([1024, 2048])
    ragged["tokens"] = min(ragged["tokens"], 4000)
    if ragged["dtype"] == "f32":
        ragged["tokens"] = min(ragged["tokens"], 1000)
    return dict(kind=kind, heads=32, kv_heads=8, dim=dim, vdim=dim,
                talk=talk, chunk=limit if talk else 0,
                window=0 if talk else limit,
                keep_first=0 if talk else rng.choice([0, 4]),
                softcap=0.0 if talk else rng.choice([0.0, 30.0]),
                ctx=_log(rng, 20, 4000), **ragged)


# ---------------------------------------------------------------------------
# shared pieces
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _lengths(case):
    """Ragged prompt lengths of the case, largest share about three times the
    smallest."""
    n, total = case["prompts"], case["tokens"]
    if not n:
        return []
    rng = random.Random(total * 131 + n)
    shares = [rng.uniform(1.0, 3.0) for _ in range(n)]
    out = [max(2, int(total * s / sum(shares))) for s in shares]
    out[0] += max(0, total - sum(out))
    return out


def _segments(case):
    """[(first row, rows, first position)] of a step: prompt portions first
    (the first one continues a prompt when `past` is given), then single
    tokens behind `past` positions."""
    segs, at = [], 0
    for i, n in enumerate(_lengths(case)):
        segs.append((at, n, case["past"] if i == 0 else 0))
        at += n
    for _ in range(case["singles"]):
        segs.append((at, 1, max(case["past"], 1)))
        at += 1
    return segs, at


def _seq_rows(segs):
    """(device rows, slots): segment i's state slot."""
    order = list(range(len(segs)))
    random.Random(len(segs) * 7 + 3).shuffle(order)
    rows = [(t0, n, p0, order[i]) for i, (t0, n, p0) in enumerate(segs)]
    return torch.tensor(rows, dtype=torch.int32, device="cuda"), rows


def _normal(gen, shape, dtype, std=1.0, mean=0.0):
    t = torch.empty(shape, dtype=dtype, device="cuda")
    return t.normal_(mean, std, generator=gen)


def _columns(proj, *widths):
    """Views of a fused projection's columns."""
    out, at = [], 0
    for w in widths:
        out.append(proj[:, at:at + w])
        at += w
    return out


def _pages(rng, lens):
    """Block tables over shuffled pages: (table int32 [S, longest], pages)."""
    need = [-(-n // BLOCK) for n in lens]
    ids = np.array(rng.sample(range(sum(need)), sum(need)), dtype=np.int32)
    table = np.zeros((len(lens), max(need)), dtype=np.int32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = ids[at:at + n]
        at += n
    return table, sum(need)


# ---------------------------------------------------------------------------
# Llama steps
# ---------------------------------------------------------------------------
def _contexts(case):
    rng = random.Random(case["seqs"] * 1009 + case["ctx_hi"])
    return [rng.randint(case["ctx_lo"], case["ctx_hi"])
            for _ in range(case["seqs"])]


def _arch(case):
    from production_stack_amd.engine.config import ARCHITECTURES

    return dataclasses.replace(ARCHITECTURES[case["arch"]],
                               num_layers=case["layers"])


def _llama_lens(case):
    """Cached positions of every sequence after the step: prompts, singles."""
    lens = []
    if case["kind"] == "mixed_step":
        lens = [n + (case["past"] if i % 2 == 0 else 0)
                for i, n in enumerate(_lengths(case))]
    return lens, _contexts(case)


def _llama_prepare(case, seed):
    from production_stack_amd import ops
    from production_stack_amd.engine.config import (
        CacheConfig,
        EngineConfig,
        SchedulerConfig,
    )
    from production_stack_amd.engine.graph_runner import DecodeGraphRunner
    from production_stack_amd.engine.model_runner import ModelRunner
    from production_stack_amd.engine.models.llama import BatchMeta

    plens, dlens = _llama_lens(case)
    table, pages = _pages(random.Random(seed), plens + dlens)
    graph = case["kind"] == "decode_step"
    cfg = EngineConfig(
        model=case["arch"], seed=int(seed), max_model_len=8192,
        cache=CacheConfig(block_size=BLOCK, num_gpu_blocks=pages,
                          kv_cache_dtype=case["kv"]),
        scheduler=SchedulerConfig(max_num_seqs=case["seqs"]))
    mcfg = _arch(case)
    runner = ModelRunner(cfg, mcfg, torch.device("cuda"))
    runner.allocate_kv_cache(pages)
    graphs = None
    if graph:
        # the graphs as the engine captures them, without its start-up timing
        # of GEMM variants: which of them wins differs from run to run
        graphs = DecodeGraphRunner(
            runner.model, runner.kv_caches, case["seqs"],
            cfg.max_model_len // BLOCK, torch.device("cuda"))
        graphs.capture_all()
    gen = _gen(seed)
    for kv in runner.kv_caches:
        for t in kv:
            if t.dtype == torch.bfloat16:
                t.normal_(0.0, 1.0, generator=gen)
            else:
                for part in t.split(4096):
                    part.copy_(_normal(gen, part.shape, torch.bfloat16))
    chunks = _lengths(case) if plens else []
    starts = [n - c for n, c in zip(plens, chunks)]
    pos = np.concatenate(
        [np.arange(s, s + c) for s, c in zip(starts, chunks)]
        + [np.array([n - 1 for n in dlens])]).astype(np.int64)
    row = np.concatenate(
        [np.full(c, i) for i, c in enumerate(chunks)]
        + [len(chunks) + np.arange(len(dlens))]).astype(np.int64)
    slots = table[row, pos // BLOCK].astype(np.int64) * BLOCK + pos % BLOCK
    tokens = torch.randint(16, mcfg.vocab_size, (len(pos),), generator=gen,
                           device="cuda")
    state = dict(case=case, runner=runner, graphs=graphs, tokens=tokens, pos=pos, row=row,
                 table=table, slots=slots, plens=plens, dlens=dlens,
                 chunks=chunks, starts=starts)
    if graph:
        state["step"] = (tokens.cpu().numpy(), pos.astype(np.int32), slots,
                         (pos + 1).astype(np.int32),
                         [table[i, :-(-n // BLOCK)].tolist()
                          for i, n in enumerate(dlens)])
        return state
    tile = ops.prefill_tile_rows(mcfg.num_q_heads, mcfg.num_kv_heads)
    tiles, at = [], 0
    for i, (s, c) in enumerate(zip(starts, chunks)):
        tiles += [(i, at + t, s + t, min(tile, c - t))
                  for t in range(0, c, tile)]
        at += c

    def dev(a, dtype=torch.int32):
        return torch.tensor(np.asarray(a), dtype=dtype, device="cuda")

    npt = at
    tab = dev(table)
    state["meta"] = BatchMeta(
        positions=dev(pos), slot_mapping=dev(slots, torch.long),
        num_prefill_tokens=npt, prefill_token_seq=dev(row[:npt]),
        prefill_token_pos=dev(pos[:npt]),
        prefill_block_tables=tab[:len(chunks)], num_decode_seqs=len(dlens),
        decode_seq_lens=dev(dlens), decode_block_tables=tab[len(chunks):],
        prefill_tiles=dev(tiles))
    # logits are wanted at the last row of every prompt and at single tokens
    last = list(np.cumsum(chunks) - 1) + list(range(npt, len(pos)))
    state["last"] = dev(last, torch.long)
    return state


def _llama_run(state):
    runner = state["runner"]
    if state["case"]["kind"] == "decode_step":
        return state["graphs"].run(*state["step"])
    hidden = runner.model(state["tokens"], state["meta"], runner.kv_caches)
    return runner.model.compute_logits(hidden[state["last"]])


def _rms64(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w.double()


def _llama_exact(case, seed):
    st = _llama_prepare(case, seed)
    model, cfg = st["runner"].model, _arch(case)
    H, G, D, F = (cfg.num_q_heads, cfg.num_kv_heads, cfg.head_dim,
                  cfg.intermediate_size)
    pos = torch.tensor(st["pos"], device="cuda")
    inv = cfg.rope_theta ** (-torch.arange(0, D, 2, dtype=torch.float64,
                                           device="cuda") / D)
    ang = pos.double().unsqueeze(1) * inv
    cos, sin = ang.cos().unsqueeze(1), ang.sin().unsqueeze(1)

    def turn(x):
        a, b = x[..., :D // 2], x[..., D // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)

    x = model.embed[st["tokens"]].double()
    T = x.shape[0]
    npt = sum(st["chunks"])
    spans = [(sum(st["chunks"][:i]), c, s) for i, (c, s) in
             enumerate(zip(st["chunks"], st["starts"]))]
    spans += [(npt + i, 1, n - 1) for i, n in enumerate(st["dlens"])]
    for layer, (kc, vc) in zip(model.layers, st["runner"].kv_caches):
        h = _rms64(x, layer.input_norm)
        qkv = h @ layer.qkv_proj.double().t()
        q = turn(qkv[:, :H * D].view(T, H, D))
        k = turn(qkv[:, H * D:(H + G) * D].view(T, G, D))
        v = qkv[:, (H + G) * D:].view(T, G, D)
        if kc.dtype != torch.bfloat16:      # what the cache would hold
            k = k.to(torch.bfloat16).to(kc.dtype).double()
            v = v.to(torch.bfloat16).to(vc.dtype).double()
        o = torch.empty(T, H, D, dtype=torch.float64, device="cuda")
        for i, (r0, n, p0) in enumerate(spans):
            ids = torch.tensor(st["table"][i, :-(-(p0 + n) // BLOCK)],
                               device="cuda").long()
            kk, vv = (c[ids].transpose(0, 1).reshape(G, -1, D)[:, :p0 + n]
                      .double() for c in (kc, vc))
            kk[:, p0:] = k[r0:r0 + n].transpose(0, 1)
            vv[:, p0:] = v[r0:r0 + n].transpose(0, 1)
            qq = (q[r0:r0 + n].transpose(0, 1)
                  .reshape(G, H // G * n, D))
            s = torch.matmul(qq, kk.transpose(1, 2)) * D ** -0.5
            s = s.view(G, H // G, n, p0 + n)
            if n > 1:
                far = (torch.arange(p0 + n, device="cuda")
                       > p0 + torch.arange(n, device="cuda").unsqueeze(1))
                s = s.masked_fill(far, float("-inf"))
            a = torch.matmul(torch.softmax(s, -1).view(G, -1, p0 + n), vv)
            o[r0:r0 + n] = a.view(H, n, D).transpose(0, 1)
        x = x + o.view(T, H * D) @ layer.o_proj.double().t()
        h = _rms64(x, layer.post_attn_norm)
        gu = h @ layer.gate_up_proj.double().t()
        x = x + ((torch.nn.functional.silu(gu[:, :F]) * gu[:, F:])
                 @ layer.down_proj.double().t())
    if "last" in st:
        x = x[st["last"]]
    return _rms64(x, model.final_norm) @ model.lm_head.double().t()


def _llama_work(case):
    cfg = _arch(case)
    plens, dlens = _llama_lens(case)
    chunks = _lengths(case) if plens else []
    H, G, D = cfg.num_q_heads, cfg.num_kv_heads, cfg.head_dim
    W, F, V = cfg.hidden_size, cfg.intermediate_size, cfg.vocab_size
    T, out = sum(chunks) + len(dlens), len(chunks) + len(dlens)
    per = W * (H + 2 * G) * D + H * D * W + 3 * W * F
    kvb = 2 * G * D * (1 if case["kv"] == "fp8" else 2)
    read = sum(dlens) + sum(plens)
    pairs = sum(dlens) + sum(c * (n - c) + c * (c + 1) / 2
                             for c, n in zip(chunks, plens))
    return {"bytes": case["layers"] * (2 * per + kvb * read) + 2 * V * W
            + 2 * T * W + 2 * out * V,
            "flops": case["layers"] * (2 * per * T + 4 * pairs * H * D)
            + 2 * out * V * W}


# ---------------------------------------------------------------------------
# recurrences
# ---------------------------------------------------------------------------
def _walk(rows, width, step):
    """Runs `step(rows of every live segment, their segments)` token by
    token over all segments at once."""
    for t in range(max(n for _, n, _, _ in rows)):
        live = [i for i, r in enumerate(rows) if r[1] > t]
        at = torch.tensor([rows[i][0] + t for i in live], device="cuda")
        step(at, torch.tensor(live, device="cuda"))


def _start64(state, rows):
    """Segment states in 64 bits, zero at position 0."""
    S = torch.stack([state[r[3]].double() for r in rows])
    for i, r in enumerate(rows):
        if r[2] == 0:
            S[i] = 0
    return S


def _put_back(state, rows, S):
    out = state.double().clone()
    for i, r in enumerate(rows):
        out[r[3]] = S[i]
    return out


def _states(gen, segs, shape, std=1.0):
    return _normal(gen, (len(segs),) + shape, torch.float32, std)


def _gdelta_prepare(case, seed):
    gen, dt = _gen(seed), _DT[case["dtype"]]
    H, D = case["heads"], case["dim"]
    HD = H * D
    segs, T = _segments(case)
    rows_t, rows = _seq_rows(segs)
    # r | k | v | g | a of one fused projection, the decay from its own
    proj = _normal(gen, (T, 5 * HD), dt)
    return dict(case=case, rows_t=rows_t, rows=rows,
                parts=_columns(proj, HD, HD, HD, HD, HD),
                zw=_normal(gen, (T, HD), dt),
                w0=_normal(gen, (HD,), torch.float32, 0.5),
                ab=_normal(gen, (HD,), torch.float32, 0.5),
                normw=_normal(gen, (HD,), torch.float32, 0.1, 1.0),
                state=_states(gen, segs, (H, D, D), 2.0))


def _gdelta_run(s):
    from production_stack_amd import ops

    r, k, v, g, za = s["parts"]
    out = ops.delta_rule(r, k, v, s["zw"], za, g, s["w0"], s["ab"],
                         s["normw"], s["state"], s["rows_t"],
                         s["case"]["heads"], EPS, math.exp(-0.5))
    return {"out": out, "state": s["state"]}


def _gdelta_exact(case, seed):
    s = _gdelta_prepare(case, seed)
    H, D = case["heads"], case["dim"]
    r, k, v, g, za = (p.double().view(-1, H, D) for p in s["parts"])
    w = torch.exp(-math.exp(-0.5) * torch.sigmoid(
        s["zw"].double() + s["w0"].double())).view(-1, H, D)
    a = torch.sigmoid(za + s["ab"].double().view(H, D))
    u = k * torch.rsqrt(k.pow(2).sum(-1, keepdim=True) + 1e-6)
    S = _start64(s["state"], s["rows"])
    o = torch.empty_like(v)

    def step(at, seg):
        old = S[seg]
        us = torch.matmul(u[at].unsqueeze(2), old)
        new = (w[at].unsqueeze(3) * old
               - (a[at] * u[at]).unsqueeze(3) * us
               + k[at].unsqueeze(3) * v[at].unsqueeze(2))
        S[seg] = new
        o[at] = torch.matmul(r[at].unsqueeze(2), new).squeeze(2)

    _walk(s["rows"], D, step)
    o = o * torch.rsqrt(o.pow(2).mean(-1, keepdim=True) + EPS)
    o = o * s["normw"].double().view(H, D) * torch.sigmoid(g)
    return {"out": o.reshape(-1, H * D),
            "state": _put_back(s["state"], s["rows"], S)}


def _gdelta_work(case):
    H, D, e = case["heads"], case["dim"], 2 if case["dtype"] == "bf16" else 4
    segs, T = _segments(case)
    carried = sum(1 for _, _, p0 in segs if p0)
    return {"bytes": T * H * D * e * 7 + (len(segs) + carried) * H * D * D * 4,
            "flops": T * H * D * D * 8.0}


def _cdelta_prepare(case, seed):
    gen, dt = _gen(seed), _DT[case["dtype"]]
    H, G, D, DV = (case["heads"], case["kv_heads"], case["dim"],
                   case["vdim"])
    segs, T = _segments(case)
    rows_t, rows = _seq_rows(segs)
    # q | k | v behind their convolution and silu
    qkv = torch.nn.functional.silu(
        _normal(gen, (T, 2 * G * D + H * DV), dt))
    return dict(case=case, rows_t=rows_t, rows=rows,
                parts=_columns(qkv, G * D, G * D, H * DV),
                beta=_normal(gen, (T, H + 256), dt)[:, :H],
                zdec=_normal(gen, (T, H * D), dt),
                zgate=_normal(gen, (T, H * DV), dt),
                a_log=torch.empty(H, device="cuda").uniform_(
                    -1.0, 1.0, generator=gen),
                dt_bias=_normal(gen, (H * D,), torch.float32, 0.5),
                normw=_normal(gen, (DV,), torch.float32, 0.1, 1.0),
                state=_states(gen, segs, (H, D, DV), 0.3))


def _cdelta_run(s):
    from production_stack_amd import ops

    q, k, v = s["parts"]
    c = s["case"]
    out = ops.gated_delta(q, k, v, s["beta"], s["zdec"], s["zgate"],
                          s["a_log"], s["dt_bias"], s["normw"], s["state"],
                          s["rows_t"], c["heads"], c["kv_heads"], EPS)
    return {"out": out, "state": s["state"]}


def _cdelta_exact(case, seed):
    s = _cdelta_prepare(case, seed)
    H, G, D, DV = (case["heads"], case["kv_heads"], case["dim"],
                   case["vdim"])
    q, k, v = (p.double() for p in s["parts"])

    def unit(x):
        x = x.view(-1, G, D)
        x = x * torch.rsqrt(x.pow(2).sum(-1, keepdim=True) + 1e-6)
        return x.repeat_interleave(H // G, dim=1)

    q, k, v = unit(q) * D ** -0.5, unit(k), v.view(-1, H, DV)
    decay = torch.exp(
        -torch.exp(s["a_log"].double()).view(H, 1)
        * torch.nn.functional.softplus(
            (s["zdec"].double() + s["dt_bias"].double()).view(-1, H, D),
            threshold=40.0))
    b = torch.sigmoid(s["beta"].double())
    S = _start64(s["state"], s["rows"])
    o = torch.empty_like(v)

    def step(at, seg):
        new = decay[at].unsqueeze(3) * S[seg]
        u = b[at].unsqueeze(2) * (
            v[at] - torch.matmul(k[at].unsqueeze(2), new).squeeze(2))
        new = new + k[at].unsqueeze(3) * u.unsqueeze(2)
        S[seg] = new
        o[at] = torch.matmul(q[at].unsqueeze(2), new).squeeze(2)

    _walk(s["rows"], D, step)
    o = o * torch.rsqrt(o.pow(2).mean(-1, keepdim=True) + EPS)
    o = (o * s["normw"].double()
         * torch.sigmoid(s["zgate"].double()).view(-1, H, DV))
    return {"out": o.reshape(-1, H * DV),
            "state": _put_back(s["state"], s["rows"], S)}


def _cdelta_work(case):
    H, G, D, DV = (case["heads"], case["kv_heads"], case["dim"],
                   case["vdim"])
    e = 2 if case["dtype"] == "bf16" else 4
    segs, T = _segments(case)
    carried = sum(1 for _, _, p0 in segs if p0)
    return {"bytes": T * e * (2 * G * D + H * D + 3 * H * DV + H)
            + (len(segs) + carried) * H * D * DV * 4,
            "flops": T * H * D * DV * 7.0}


def _scan_prepare(case, seed):
    gen, dt = _gen(seed), _DT[case["dtype"]]
    mode, H, G, D, DV = (case["mode"], case["heads"], case["groups"],
                         case["dim"], case["vdim"])
    segs, T = _segments(case)
    rows_t, rows = _seq_rows(segs)
    f32 = torch.float32
    s = dict(case=case, rows_t=rows_t, rows=rows, wr=None, p1=None, p2=None,
             normw=None, aux=None, c0=1.0, qscale=D ** -0.5,
             state=_states(gen, segs, (H, D, DV)))
    if mode == "ssd":
        # x | B | C behind the convolution and silu; z and dt are columns of
        # the input projection
        inner = H * DV
        xbc = torch.nn.functional.silu(
            _normal(gen, (T, inner + 2 * G * D), dt))
        s["v"], s["k"], s["q"] = _columns(xbc, inner, G * D, G * D)
        proj = _normal(gen, (T, inner + H), dt)
        s["gate"], s["dec"] = _columns(proj, inner, H)
        s["p0"] = _normal(gen, (H,), f32, 0.5)
        s["p1"] = torch.empty(H, device="cuda").uniform_(-1.0, 1.0,
                                                         generator=gen)
        s["p2"] = _normal(gen, (H,), f32, 0.2, 1.0)
        s["qscale"] = 1.0
        return s
    extra = 2 * H if mode == "mlstm" else 16
    proj = _normal(gen, (T, 2 * H * D + 2 * H * DV + extra), dt)
    s["q"], s["k"], s["v"], s["gate"], rest = _columns(
        proj, H * D, H * D, H * DV, H * DV, extra)
    if mode == "gla":
        s["dec"] = _normal(gen, (T, H * D), dt)
        s["p0"] = _normal(gen, (H * D,), f32, 0.5)
        s["normw"] = _normal(gen, (DV,), f32, 0.1, 1.0)
        s["c0"] = 1.0 / 16.0
    else:
        s["wr"], s["dec"] = _columns(rest, H, H)
        s["p0"] = _normal(gen, (H,), f32, 0.5)
        s["p1"] = _normal(gen, (H,), f32, 0.5, 3.0)
        s["normw"] = _normal(gen, (H * DV,), f32, 0.1, 1.0)
        s["c0"] = 15.0
        s["aux"] = _states(gen, segs, (H, D + 1))
    return s


def _scan_run(s):
    from production_stack_amd import ops

    c = s["case"]
    out = ops.linear_scan(
        c["mode"], s["q"], s["k"], s["v"], s["dec"], s["gate"], s["state"],
        s["rows_t"], c["heads"], c["groups"], EPS, qscale=s["qscale"],
        c0=s["c0"], wr=s["wr"], p0=s["p0"], p1=s["p1"], p2=s["p2"],
        normw=s["normw"], aux=s["aux"])
    got = {"out": out, "state": s["state"]}
    if s["aux"] is not None:
        got["aux"] = s["aux"]
    return got


def _scan_exact(case, seed):
    s = _scan_prepare(case, seed)
    mode, H, G, D, DV = (case["mode"], case["heads"], case["groups"],
                         case["dim"], case["vdim"])
    rows = s["rows"]

    def heads(x):
        return x.double().view(-1, G, D).repeat_interleave(H // G, dim=1)

    q, k = heads(s["q"]) * s["qscale"], heads(s["k"])
    v = s["v"].double().reshape(-1, H, DV)
    gate = s["gate"].double().reshape(-1, H, DV)
    dec, p0 = s["dec"].double(), s["p0"].double()
    S = _start64(s["state"], rows)
    o = torch.empty_like(v)
    if mode == "gla":
        a = torch.exp(torch.nn.functional.logsigmoid(dec + p0) * s["c0"])
        a = a.view(-1, H, D, 1)
        w = None
    elif mode == "ssd":
        w = torch.nn.functional.softplus(dec + p0, threshold=40.0)
        a = torch.exp(-torch.exp(s["p1"].double()) * w).view(-1, H, 1, 1)
    else:
        cap = s["c0"]
        ig = cap * torch.tanh((s["wr"].double() + p0) / cap)
        fg = torch.nn.functional.logsigmoid(
            cap * torch.tanh((dec + s["p1"].double()) / cap))
        N = _start64(s["aux"], rows)        # [S, H, D + 1]: normaliser, max

    def step(at, seg):
        kk, den = k[at], None
        if mode == "mlstm":
            m = N[seg][:, :, D]
            mn = torch.maximum(fg[at] + m, ig[at])
            at_a = torch.exp(fg[at] + m - mn)
            kk = torch.exp(ig[at] - mn).unsqueeze(2) * kk
            nn_ = at_a.unsqueeze(2) * N[seg][:, :, :D] + kk
            N[seg] = torch.cat([nn_, mn.unsqueeze(2)], dim=2)
            den = torch.maximum((nn_ * q[at]).sum(-1).abs(),
                                torch.exp(-mn)) + 1e-6
            at_a = at_a[..., None, None]
        else:
            at_a = a[at]
            if w is not None:
                kk = w[at].unsqueeze(2) * kk
        new = at_a * S[seg] + kk.unsqueeze(3) * v[at].unsqueeze(2)
        S[seg] = new
        y = torch.matmul(q[at].unsqueeze(2), new).squeeze(2)
        o[at] = y if den is None else y / den.unsqueeze(2)

    _walk(rows, D, step)
    if mode == "ssd":
        o = ((o + s["p2"].double().view(H, 1) * v)
             * torch.nn.functional.silu(gate))
    else:
        o = o * torch.rsqrt(o.pow(2).mean(-1, keepdim=True) + EPS)
        if mode == "gla":
            o = (o * s["normw"].double()
                 * torch.nn.functional.silu(gate))
        else:
            o = (o * s["normw"].double().view(H, DV) * torch.sigmoid(gate))
    got = {"out": o.reshape(-1, H * DV),
           "state": _put_back(s["state"], rows, S)}
    if mode == "mlstm":
        got["aux"] = _put_back(s["aux"], rows, N)
    return got


def _scan_work(case):
    mode, H, G, D, DV = (case["mode"], case["heads"], case["groups"],
                         case["dim"], case["vdim"])
    e = 2 if case["dtype"] == "bf16" else 4
    segs, T = _segments(case)
    carried = sum(1 for _, _, p0 in segs if p0)
    cols = 2 * G * D + 2 * H * DV + (H * D if mode == "gla" else H)
    return {"bytes": T * (e * cols + H * DV * (4 if mode == "ssd" else e))
            + (len(segs) + carried) * H * D * DV * 4,
            "flops": T * H * D * DV * 5.0}


# ---------------------------------------------------------------------------
# attention with head mix / windows
# ---------------------------------------------------------------------------
def _attn_spans(case):
    segs, T = _segments(dict(case, past=0))
    spans, i = [], 0
    rng = random.Random(case["ctx"] * 31 + case["singles"])
    for t0, n, _ in segs:
        if n > 1 or i < case["prompts"]:
            p0 = case["past"] if i == 0 else 0
        else:
            p0 = rng.randint(case["ctx"] // 2, case["ctx"] * 3 // 2)
        spans.append((t0, n, p0))
        i += 1
    return spans, T


def _attn_prepare(case, seed):
    gen, dt = _gen(seed), _DT[case["dtype"]]
    H, G, D, DV = (case["heads"], case["kv_heads"], case["dim"],
                   case["vdim"])
    spans, T = _attn_spans(case)
    table, pages = _pages(random.Random(seed), [p + n for _, n, p in spans])
    proj = _normal(gen, (T, H * D + 2 * G * D), dt)
    tok_seq = np.repeat(np.arange(len(spans)), [n for _, n, _ in spans])
    tok_pos = np.concatenate([np.arange(p, p + n) for _, n, p in spans])

    def dev(a):
        return torch.tensor(a, dtype=torch.int32, device="cuda")

    talk = sinks = None
    if case["talk"]:
        talk = _normal(gen, (H, H), torch.float32, 0.2)
        talk += torch.eye(H, device="cuda")
    else:
        sinks = _normal(gen, (H,), torch.float32, 0.5)
    return dict(case=case, q=proj[:, :H * D], spans=spans, table=table,
                table_t=dev(table), seq=dev(tok_seq), pos=dev(tok_pos),
                npt=sum(n for _, n, _ in spans if n > 1), T=T, talk=talk,
                sinks=sinks,
                k=_normal(gen, (pages, G, BLOCK, D), dt),
                v=_normal(gen, (pages, G, BLOCK, DV), dt))


def _attn_run(s):
    from production_stack_amd import ops

    c, npt, T = s["case"], s["npt"], s["T"]
    H = c["heads"]
    out = torch.empty((T, H * c["vdim"]), dtype=s["q"].dtype, device="cuda")
    # prompt portions and single tokens are two calls, as in the layers
    for a, b, variant in ((0, npt, 0), (npt, T, 3)):
        if b > a:
            ops.talk_attention(
                s["q"][a:b], s["k"], s["v"], s["table_t"], s["seq"][a:b],
                s["pos"][a:b], c["dim"] ** -0.5, H, chunk=c["chunk"],
                window=c["window"], sink=True, talk=s["talk"],
                out=out[a:b], variant=variant, keep_first=c["keep_first"],
                softcap=c["softcap"], sink_vals=s["sinks"])
    return out


def _attn_exact(case, seed):
    s = _attn_prepare(case, seed)
    H, G, D, DV = (case["heads"], case["kv_heads"], case["dim"],
                   case["vdim"])
    q = s["q"].double().view(-1, H, D)
    out = torch.empty(s["T"], H, DV, dtype=torch.float64, device="cuda")
    sink = (s["sinks"].double() if s["sinks"] is not None
            else torch.zeros(H, dtype=torch.float64, device="cuda"))
    for i, (t0, n, p0) in enumerate(s["spans"]):
        ids = torch.tensor(s["table"][i, :-(-(p0 + n) // BLOCK)],
                           device="cuda").long()
        kk, vv = (c[ids].transpose(0, 1).reshape(G, ids.numel() * BLOCK, -1)
                  [:, :p0 + n].double() for c in (s["k"], s["v"]))
        for b in range(0, n, 256):
            m = min(256, n - b)
            qq = q[t0 + b:t0 + b + m].transpose(0, 1)       # [H, m, D]
            sc = torch.matmul(qq.reshape(G, -1, D), kk.transpose(1, 2))
            sc = sc.view(H, m, p0 + n) * D ** -0.5
            if s["talk"] is not None:
                sc = torch.matmul(s["talk"].double(),
                                  sc.view(H, -1)).view(H, m, p0 + n)
            if case["softcap"]:
                sc = case["softcap"] * torch.tanh(sc / case["softcap"])
            pos = p0 + b + torch.arange(m, device="cuda").unsqueeze(1)
            key = torch.arange(p0 + n, device="cuda")
            seen = key <= pos
            if case["chunk"]:
                seen &= key >= pos // case["chunk"] * case["chunk"]
            if case["window"]:
                seen &= ((pos - key < case["window"])
                         | (key < case["keep_first"]))
            sc = sc.masked_fill(~seen, float("-inf"))
            sc = torch.cat([sc, sink.view(H, 1, 1).expand(H, m, 1)], dim=2)
            p = torch.softmax(sc, -1)[..., :-1]
            o = torch.matmul(p.reshape(G, -1, p0 + n), vv)
            out[t0 + b:t0 + b + m] = o.view(H, m, DV).transpose(0, 1)
    return out.view(s["T"], H * DV)


def _attn_work(case):
    H, G, D, DV = (case["heads"], case["kv_heads"], case["dim"],
                   case["vdim"])
    e = 2 if case["dtype"] == "bf16" else 4
    spans, T = _attn_spans(case)
    pairs = keys = 0
    for _, n, p0 in spans:
        pos = np.arange(p0, p0 + n)
        lo = np.zeros_like(pos)
        if case["chunk"]:
            lo = pos // case["chunk"] * case["chunk"]
        if case["window"]:
            lo = np.maximum(lo, pos - case["window"] + 1)
        pairs += int((pos - lo + 1 + np.minimum(case["keep_first"], lo)).sum())
        keys += int(p0 + n - lo[0])
    per = 2 * H * (D + DV) + (2 * H * H if case["talk"] else 0)
    return {"bytes": e * (T * H * (D + DV) + keys * G * (D + DV)),
            "flops": float(pairs) * per}


# ---------------------------------------------------------------------------
# routed experts
# ---------------------------------------------------------------------------
LIMIT = 7.0


def _experts_prepare(case, seed):
    gen, bf = _gen(seed), torch.bfloat16
    W, F, E = case["width"], case["ff"], case["experts"]
    return dict(case=case, x=_normal(gen, (case["rows"], W), bf),
                router=_normal(gen, (E, W), bf, W ** -0.5),
                w_in=_normal(gen, (E, 2 * F, W), bf, W ** -0.5),
                w_out=_normal(gen, (E, W, F), bf, F ** -0.5))


def _experts_run(s):
    from production_stack_amd import ops

    c, x = s["case"], s["x"]
    w, sel, _ = ops.moe_route(x, s["router"], c["top"], c["score"],
                              c["score"] == "softmax")
    offs, rows, pos = ops.expert_plan(sel, c["experts"])
    ys = ops.experts_grouped(x, s["w_in"], s["w_out"], offs, rows, c["act"],
                             LIMIT)
    out = ops.experts_sum(ys, pos, c["top"], w, 1.0, None, c["experts"], x)
    return {"out": out, "weights": w, "sel": sel}


def _experts_exact(case, seed):
    s = _experts_prepare(case, seed)
    x, F = s["x"].double(), case["ff"]
    logits = x @ s["router"].double().t()
    score = (torch.softmax(logits, -1) if case["score"] == "softmax"
             else torch.sigmoid(logits))
    sel = torch.topk(logits, case["top"], dim=-1).indices
    w = score.gather(1, sel)
    if case["score"] == "softmax":
        w = w / w.sum(-1, keepdim=True)
    out = torch.zeros_like(x)
    for e in range(case["experts"]):
        gu = x @ s["w_in"][e].double().t()
        g, u = gu[:, :F], gu[:, F:]
        if case["act"] == "silu":
            act = torch.nn.functional.silu(g) * u
        else:
            g = g.clamp(max=LIMIT)
            act = (g * torch.sigmoid(1.702 * g)
                   * (u.clamp(-LIMIT, LIMIT) + 1.0))
        mine = (w * (sel == e)).sum(-1, keepdim=True)
        out += mine * (act @ s["w_out"][e].double().t())
    return {"out": out, "weights": w, "sel": None}


def _experts_work(case):
    W, F, E, n = case["width"], case["ff"], case["experts"], case["rows"]
    used = E * (1.0 - (1.0 - case["top"] / E) ** n)     # experts hit
    return {"bytes": used * 6.0 * W * F + 2 * E * W + n * W * 6,
            "flops": 6.0 * n * case["top"] * W * F + 2 * n * W * E}


# ---------------------------------------------------------------------------
# entry points
# ---------------------------------------------------------------------------
_KINDS = {
    "decode_step": (_llama_prepare, _llama_run, _llama_exact, _llama_work),
    "mixed_step": (_llama_prepare, _llama_run, _llama_exact, _llama_work),
    "general_delta": (_gdelta_prepare, _gdelta_run, _gdelta_exact,
                      _gdelta_work),
    "channel_delta": (_cdelta_prepare, _cdelta_run, _cdelta_exact,
                      _cdelta_work),
    "scan": (_scan_prepare, _scan_run, _scan_exact, _scan_work),
    "attention": (_attn_prepare, _attn_run, _attn_exact, _attn_work),
    "experts": (_experts_prepare, _experts_run, _experts_exact,
                _experts_work),
}


def prepare(case, seed):
    with torch.no_grad():
        return _KINDS[case["kind"]][0](case, seed)


def run(state):
    with torch.no_grad():
        return _KINDS[state["case"]["kind"]][1](state)


def exact(case, seed):
    with torch.no_grad():
        return _KINDS[case["kind"]][2](case, seed)


def work(case):
    return _KINDS[case["kind"]][3](case)


def tolerance(case):
    if case["kind"] in ("decode_step", "mixed_step"):
        # bf16 activations rounded between the products of several layers:
        # 0.01 to 0.02 from the 64-bit logits after 2 to 8 layers
        return {"rel": 0.03, "max": 0.3}
    if case["kind"] == "experts":
        # 0.0035 measured: bf16 between the two products
        return {"rel": 0.01, "max": 0.1, "differ": 0.01}
    if case.get("dtype") == "f32":
        return {"rel": 2e-5, "max": 2e-3}
    # bf16 results of fp32 arithmetic, 0.0017 measured; the largest
    # difference is one rounding step of a large value
    return {"rel": 0.004, "max": 0.02}
