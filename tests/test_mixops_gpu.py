"""HIP kernels of the fp32-residual / delta-rule / talking-attention ops
against their plain PyTorch fp32 references (production_stack_amd.ops.
reference), in bfloat16 and float32, on shapes that exercise padding,
strided views, page borders, chunk/window edges and slot reuse."""

import math

import pytest
import torch

from production_stack_amd import ops
from production_stack_amd.ops import reference

pytestmark = pytest.mark.gpu

DTYPES = [torch.bfloat16, torch.float32]


def tol(dtype):
    return dict(rtol=2e-2, atol=2e-2) if dtype == torch.bfloat16 else dict(
        rtol=2e-5, atol=2e-5)


def test_native_library_loaded():
    from production_stack_amd.ops import native

    assert native.load() is not None


class _Launches:
    """The library, with the arguments of the calls that were made."""

    def __init__(self, lib):
        self.lib, self.made = lib, []

    def __getattr__(self, name):
        fn = getattr(self.lib, name)

        def call(*args):
            self.made.append((name, args))
            return fn(*args)

        return call

    def shares(self):
        return self.made[-1][1][-3]       # ahead of the records and the stream


@pytest.mark.parametrize("dtype", DTYPES)
def test_embed_scale(dtype):
    g = torch.Generator().manual_seed(0)
    emb = torch.randn(97, 200, generator=g).to(dtype)
    tok = torch.randint(0, 97, (33,), generator=g)
    want = reference.embed_scale(tok, emb, 3.25)
    got = ops.embed_scale(tok.cuda(), emb.cuda(), 3.25)
    assert got.dtype == torch.float32
    torch.testing.assert_close(got.cpu(), want, rtol=0, atol=0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("ndelta", [0, 1, 2])
def test_add_rms_norm32(dtype, ndelta):
    g = torch.Generator().manual_seed(1)
    T, W = 19, 328
    x = torch.randn(T, W, generator=g) * 3
    w = torch.randn(W, generator=g)
    deltas = [torch.randn(T, W, generator=g).to(dtype)
              for _ in range(ndelta)]
    xr = x.clone()
    want = reference.add_rms_norm32(xr, deltas, w, 1e-5, dtype)
    xg = x.cuda()
    got = ops.add_rms_norm32(xg, [d.cuda() for d in deltas], w.cuda(), 1e-5,
                             dtype)
    torch.testing.assert_close(xg.cpu(), xr, rtol=1e-6, atol=1e-6)
    torch.testing.assert_close(got.cpu().float(), want.float(), **tol(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("kind,limit", [("silu", 0.0), ("gelu_tanh", 0.0),
                                        ("clamped_swish", 1.25)])
def test_gated_act_strided(dtype, kind, limit):
    g = torch.Generator().manual_seed(2)
    T, F = 11, 300
    proj = (torch.randn(T, 2 * F + 7, generator=g) * 2).to(dtype)
    want = reference.gated_act(proj[:, 3:3 + F], proj[:, 3 + F:3 + 2 * F],
                               kind, limit, dtype)
    pg = proj.cuda()
    buf = torch.zeros(T, F + 5, dtype=dtype, device="cuda")
    ops.gated_act(pg[:, 3:3 + F], pg[:, 3 + F:3 + 2 * F], kind, limit,
                  out=buf[:, 5:])
    torch.testing.assert_close(buf[:, 5:].cpu().float(), want.float(),
                               **tol(dtype))
    assert float(buf[:, :5].abs().sum()) == 0.0


def _paged(T_total, G, D, DV, bs, dtype, gen, n_seqs):
    """Random paged caches with scattered, non-monotonic block tables."""
    per = (T_total + bs - 1) // bs
    nb = per * n_seqs + 3
    perm = torch.randperm(nb, generator=gen)
    tables = perm[: per * n_seqs].view(n_seqs, per).to(torch.int32)
    kc = torch.randn(nb, G, bs, D, generator=gen).to(dtype)
    vc = torch.randn(nb, G, bs, DV, generator=gen).to(dtype)
    return kc, vc, tables


@pytest.mark.parametrize("dtype", DTYPES)
def test_kv_append_distinct_widths(dtype):
    g = torch.Generator().manual_seed(3)
    G, D, DV, bs = 3, 40, 24, 16
    kc, vc, tables = _paged(50, G, D, DV, bs, dtype, g, 1)
    T = 21
    proj = torch.randn(T, G * D + G * DV + 9, generator=g).to(dtype)
    pos = torch.arange(7, 7 + T)
    slots = tables[0].long()[pos // bs] * bs + pos % bs
    kr, vr = kc.clone(), vc.clone()
    reference.kv_append(proj[:, 4:4 + G * D].reshape(T, G, D),
                        proj[:, 4 + G * D:4 + G * D + G * DV].reshape(
                            T, G, DV), kr, vr, slots)
    kg, vg, pg = kc.cuda(), vc.cuda(), proj.cuda()
    ops.kv_append(pg[:, 4:4 + G * D], pg[:, 4 + G * D:4 + G * D + G * DV],
                  kg, vg, slots.cuda())
    assert torch.equal(kg.cpu(), kr) and torch.equal(vg.cpu(), vr)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("variant", [1, 2, 4, 41, 43])
@pytest.mark.parametrize("H,G,D,DV,chunk,window,sink,talk", [
    (4, 2, 40, 40, 24, 0, True, True),
    (6, 3, 40, 24, 40, 0, True, True),
    (3, 1, 32, 64, 0, 0, False, False),
    (4, 4, 16, 16, 0, 20, True, False),
    (8, 2, 64, 32, 37, 0, False, True),
    (32, 8, 128, 128, 64, 0, True, True),
    (16, 4, 72, 96, 0, 50, True, True),
    (5, 5, 24, 24, 30, 0, True, True),
])
def test_talk_attention(dtype, variant, H, G, D, DV, chunk, window, sink,
                        talk):
    g = torch.Generator().manual_seed(4)
    bs, n_seqs, L = 16, 3, 150
    kc, vc, tables = _paged(L, G, D, DV, bs, dtype, g, n_seqs)
    # ragged batch: a long portion, a portion crossing chunk/page edges,
    # single tokens at edges
    token_seq, token_pos = [], []
    for s, (a, b) in enumerate([(0, 70), (90, 131), (149, 150)]):
        token_seq += [s] * (b - a)
        token_pos += list(range(a, b))
    edge = chunk or window or bs
    for p in (edge - 1, edge, edge + 1, 2 * edge - 1, 2 * edge):
        token_seq.append(1)
        token_pos.append(p)
    # single tokens of different sequences side by side (decode rows)
    for s, p in ((0, 69), (2, 149), (1, 130), (2, 0), (0, 0), (1, 1)):
        token_seq.append(s)
        token_pos.append(p)
    T = len(token_seq)
    q = torch.randn(T, H * D + 5, generator=g).to(dtype)
    tk = (torch.eye(H) + 0.3 * torch.randn(H, H, generator=g)) if talk \
        else None
    ts = torch.tensor(token_seq, dtype=torch.int32)
    tp = torch.tensor(token_pos, dtype=torch.int32)
    scale = 1.0 / math.sqrt(D)
    want = reference.talk_attention(
        q[:, :H * D].float().reshape(T, H, D), kc.float(), vc.float(),
        tables, ts, tp, scale, chunk, window, sink, tk)
    got = ops.talk_attention(
        q.cuda()[:, :H * D], kc.cuda(), vc.cuda(), tables.cuda(), ts.cuda(),
        tp.cuda(), scale, H, chunk=chunk, window=window, sink=sink,
        talk=tk.cuda() if tk is not None else None,
        # 41 / 43: the split-key kernel with one / three workgroups a token
        variant=min(variant, 4), splits=variant - 40 if variant > 4 else 0)
    torch.testing.assert_close(got.cpu().float().view(T, H, DV), want,
                               **tol(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,D", [(2, 56), (3, 16), (1, 72), (2, 128),
                                 (1, 160)])
def test_delta_rule(dtype, H, D):
    g = torch.Generator().manual_seed(5)
    HD = H * D
    slots = 5
    # segments: fresh long one (tile remainder), continuing ones (slot
    # state kept), a fresh single token in a slot holding stale state
    segs = [(0, 37, 0, 3), (37, 1, 9, 1), (38, 18, 4, 0), (56, 1, 0, 4),
            (57, 2, 100, 2)]
    T = 59
    proj = torch.randn(T, 6 * HD + 3, generator=g).to(dtype)
    views = [proj[:, i * HD:(i + 1) * HD] for i in range(6)]
    w0 = torch.randn(HD, generator=g)
    ab = torch.randn(HD, generator=g)
    nw = torch.randn(HD, generator=g)
    state = torch.randn(slots, H, D, D, generator=g) * 0.3
    rows = torch.tensor(segs, dtype=torch.int32)
    sr = state.clone()
    sh = (T, H, D)
    want = reference.delta_rule(
        *[v.float().reshape(sh) for v in views], w0, ab, nw, sr, rows,
        1e-5, 0.6, torch.float32)
    sg = state.cuda()
    pg = proj.cuda()
    gviews = [pg[:, i * HD:(i + 1) * HD] for i in range(6)]
    got = ops.delta_rule(*gviews, w0.cuda(), ab.cuda(), nw.cuda(), sg,
                         rows.cuda(), H, 1e-5, 0.6)
    t = tol(dtype)
    torch.testing.assert_close(got.cpu().float().view(sh), want, **t)
    torch.testing.assert_close(sg.cpu(), sr, rtol=1e-4, atol=1e-4)


def _recurrence(mode, H, D, DV, segs, dtype, seed=0):
    """(inputs, state, aux, call): call(inputs, state, aux, rows) runs one of
    the five recurrences on the tensors' device."""
    g = torch.Generator().manual_seed(seed)
    T = sum(n for _, n, _, _ in segs)
    G = H if mode in ("general", "gla", "mlstm") else max(1, H // 2)
    dim = {"q": G * D, "k": G * D, "v": H * DV, "gate": H * DV}
    dim["dec"] = H * D if mode in ("general", "channel", "gla") else H
    dim["a"] = H * D if mode == "general" else H
    # one fused buffer, odd row stride: views as a projection leaves them
    proj = torch.randn(T, sum(dim.values()) + 3, generator=g).to(dtype)
    x, at = {}, 0
    for k, n in dim.items():
        x[k], at = proj[:, at:at + n], at + n
    x["p0"] = torch.randn(dim["dec"], generator=g) * 0.5
    x["p1"] = torch.randn(dim["a"], generator=g) * 0.5
    x["p2"] = torch.randn(H, generator=g)
    x["nw"] = torch.randn(
        H * DV if mode in ("general", "mlstm") else DV, generator=g)
    state = torch.randn(len(segs), H, D, DV, generator=g) * 0.3
    aux = None
    if mode == "mlstm":
        aux = torch.randn(len(segs), H, D + 1, generator=g).abs()

    def call(x, state, aux, rows):
        if mode == "general":
            return ops.delta_rule(x["q"], x["k"], x["v"], x["dec"], x["a"],
                                  x["gate"], x["p0"], x["p1"], x["nw"],
                                  state, rows, H, 1e-5, 0.6)
        if mode == "channel":
            return ops.gated_delta(x["q"], x["k"], x["v"], x["a"], x["dec"],
                                   x["gate"], x["p1"], x["p0"], x["nw"],
                                   state, rows, H, G, 1e-5)
        return ops.linear_scan(
            mode, x["q"], x["k"], x["v"], x["dec"], x["gate"], state, rows,
            H, G, 1e-5, qscale=D ** -0.5, c0=5.0 if mode == "mlstm" else 0.1,
            wr=x["a"] if mode == "mlstm" else None, p0=x["p0"], p1=x["p1"],
            p2=x["p2"], normw=x["nw"], aux=aux)

    return x, state, aux, call


def _to_gpu(x):
    # keep the views' strides
    base = x["q"]._base.cuda()
    return {k: (torch.as_strided(base, v.shape, v.stride(),
                                 v.storage_offset())
                if v._base is not None else v.cuda()) for k, v in x.items()}


def _rel(a, b):
    a, b = a.double().cpu(), b.double().cpu()
    return ((a - b).norm() / b.norm()).item()


def _segs(lens, starts):
    rows, at = [], 0
    for i, (n, p) in enumerate(zip(lens, starts)):
        rows.append((at, n, p, len(lens) - 1 - i))
        at += n
    return rows


RECURRENCES = ["general", "channel", "gla", "ssd", "mlstm"]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("mode", RECURRENCES)
@pytest.mark.parametrize("H,D,DV", [
    (2, 20, 20), (2, 32, 32), (4, 48, 33), (2, 64, 96), (2, 96, 64),
    (2, 128, 128), (2, 100, 160), (2, 128, 256)])
def test_recurrence_chunk_edges(mode, H, D, DV, dtype):
    """Segments of 15, 16, 17 ... rows (below, at and past whole chunks),
    single rows between them, fresh and continued, on permuted slots."""
    if mode == "general":
        DV = D
    rows = _segs([17, 1, 16, 15, 32, 2, 49, 1, 33],
                 [0, 7, 5, 3, 0, 0, 9, 0, 1])
    x, state, aux, call = _recurrence(mode, H, D, DV, rows, dtype)
    # descending order of the rows: nothing may depend on it
    rows = torch.tensor(rows[::-1], dtype=torch.int32)
    sg = state.cuda()
    ag = aux.cuda() if aux is not None else None
    got = call(_to_gpu(x), sg, ag, rows.cuda())
    want = call(x, state, aux, rows)
    # fp32 sums of up to 49 tokens x 128 channels, then one rounding
    assert _rel(got, want) < (2e-5 if dtype == torch.float32 else 6e-3)
    assert _rel(sg, state) < 2e-6
    if aux is not None:
        assert _rel(ag, aux) < 2e-6


@pytest.mark.parametrize("bad_row", [5, 21])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("mode", RECURRENCES)
@pytest.mark.parametrize("D", [32, 64, 96, 128])
def test_recurrence_chunk_not_a_number(mode, dtype, bad_row, D):
    """A value, key or decay that is no number reaches no earlier row, not
    even of its own chunk, and no other sequence."""
    rows = _segs([40, 33], [0, 4])
    x, state, aux, call = _recurrence(mode, 2, D, D, rows, dtype)
    rows = torch.tensor(rows, dtype=torch.int32).cuda()
    xg = _to_gpu(x)
    clean = call(xg, state.cuda(), aux.cuda() if aux is not None else None,
                 rows)
    for name, bad in (("v", float("nan")), ("v", float("inf")),
                      ("k", float("nan")), ("dec", float("nan"))):
        y = _to_gpu(x)
        y[name][bad_row, min(3, y[name].shape[1] - 1)] = bad
        got = call(y, state.cuda(), aux.cuda() if aux is not None else None,
                   rows)
        # other sums within the chunk; rows of bf16 round once more
        near = 1e-6 if got.dtype == torch.float32 else 2 ** -9
        assert _rel(got[:bad_row], clean[:bad_row]) < near, name
        assert _rel(got[40:], clean[40:]) < 1e-6, name
        assert not torch.isfinite(got[bad_row:40]).all(), name


def test_recurrence_chunk_exactness():
    """Rows of the state-space scan of bf16 rows against 64 bits: no further from
    them than sums of fp32 products are (1.055e-7 for these inputs, 9.8e-8 here;
    the state 6.3e-8 for 7.5e-8)."""
    H, G, D, DV, T = 48, 6, 128, 64, 700
    g = torch.Generator(device="cuda").manual_seed(1)
    act = torch.nn.functional.silu(torch.randn(
        T, H * DV + 2 * G * D, generator=g, device="cuda").to(torch.bfloat16))
    v, k, q = act.split([H * DV, G * D, G * D], dim=1)
    proj = torch.randn(T, H * DV + H, generator=g, device="cuda").to(
        torch.bfloat16)
    gate, dec = proj.split([H * DV, H], dim=1)
    p0, p1, p2 = (torch.randn(H, generator=g, device="cuda") * 0.4
                  for _ in range(3))
    state = torch.randn(1, H, D, DV, generator=g, device="cuda")
    S = state[0].double()
    rows = torch.tensor([[0, T, 1, 0]], dtype=torch.int32, device="cuda")
    got = ops.linear_scan("ssd", q, k, v, dec, gate, state, rows, H, G, 1e-5,
                          p0=p0, p1=p1, p2=p2)
    w = torch.nn.functional.softplus(dec.double() + p0.double(),
                                     threshold=40.0)
    a = torch.exp(-torch.exp(p1.double()) * w)
    q, k = (x.double().view(T, G, D).repeat_interleave(H // G, dim=1)
            for x in (q, k))
    vd = v.double().reshape(T, H, DV)
    want = torch.empty_like(vd)
    for t in range(T):
        S = a[t].view(H, 1, 1) * S + (w[t].view(H, 1) * k[t]).unsqueeze(
            2) * vd[t].unsqueeze(1)
        want[t] = (S * q[t].unsqueeze(2)).sum(1)
    want = ((want + p2.double().view(H, 1) * vd)
            * torch.nn.functional.silu(gate.double().reshape(T, H, DV)))
    assert _rel(got, want.reshape(T, H * DV)) < 1.05e-7
    assert _rel(state[0], S) < 7.5e-8


@pytest.mark.parametrize("lens,tokens", [
    ([75, 33], (5, 21, 37, 64, 74)), ([700], (100, 351))])
@pytest.mark.parametrize("D", [32, 64, 96, 128])
@pytest.mark.parametrize("mode", ["ssd", "mlstm"])
def test_recurrence_chunk_infinities(mode, D, lens, tokens):
    """Values, keys, queries and states that are infinite, or no numbers, in
    either half of a chunk of 32 and in one of several runs: bf16 rows leave
    infinities and not-a-numbers in the state where fp32 rows of the same values
    do, whose products are made as they are (k inf is an infinity). Earlier rows
    and other sequences stay as they are."""
    H, DV = 2, 40
    segs = _segs(lens, [3, 4])
    x, state, aux, call = _recurrence(mode, H, D, DV, segs, torch.bfloat16)
    rows = torch.tensor(segs, dtype=torch.int32).cuda()
    base = x["q"]._base.float()
    wide = {k: (torch.as_strided(base, v.shape, v.stride(),
                                 v.storage_offset())
                if v._base is not None else v) for k, v in x.items()}

    def run(x, name, at, bad):
        x, st = _to_gpu(x), state.clone()
        if name == "state":  # one entry, which every row of its head meets
            st[segs[0][3], at % H, 5, 3] = bad
        elif name:
            x[name][at, 3] = bad
        st = st.cuda()
        ax = aux.cuda() if aux is not None else None
        out = call(x, st, ax, rows)
        return [t.float() for t in (out, st, ax) if t is not None]

    def same(a, b):
        for what in (math.inf, -math.inf):
            assert torch.equal(a == what, b == what)
        assert torch.equal(a.isnan(), b.isnan())

    clean = run(x, None, 0, 0.0)
    near = 1e-6 if mode == "ssd" else 2 ** -9  # other sums, one rounding
    # (decays over a run may come to zero, which leaves no infinity)
    for name in ("v", "k", "q") + (("state",) if len(lens) > 1 else ()):
        for at in tokens:
            for bad in (math.inf, -math.inf, math.nan):
                got, want = run(x, name, at, bad), run(wide, name, at, bad)
                for a, b in zip(got[1:], want[1:]):
                    same(a, b)
                if name == "state":
                    same(got[0], want[0])
                else:
                    # sums of several infinities: which chunk they meet in
                    # says whether they come to one or to none
                    assert not got[0][at, 3].isfinite()
                    assert _rel(got[0][:at], clean[0][:at]) < near
                assert torch.equal(got[0][lens[0]:], clean[0][lens[0]:])
                # numbers stay: one rounding to bf16, states are fp32
                for a, b, c in zip(got, want, (6e-3, 2e-6, 2e-6)):
                    ok = a.isfinite() & b.isfinite()
                    assert not ok.any() or _rel(a[ok], b[ok]) < c


@pytest.mark.parametrize("mode", ["general", "channel", "gla"])
def test_recurrence_chunk_fast_decay(mode):
    """Decays whose product over half a chunk leaves fp32's range: ratios of
    neighbouring tokens stay exact."""
    rows = _segs([50, 16], [0, 4])
    x, state, aux, call = _recurrence(mode, 2, 64, 64, rows, torch.float32)
    if mode == "channel":
        x["p1"] += 3.0                  # rates around 20
    elif mode == "gla":
        x["p0"] -= 150.0                # logs around -15
    else:
        def call(x, state, aux, rows):
            return ops.delta_rule(x["q"], x["k"], x["v"], x["dec"], x["a"],
                                  x["gate"], x["p0"], x["p1"], x["nw"],
                                  state, rows, 2, 1e-5, 40.0)

    rows = torch.tensor(rows, dtype=torch.int32)
    sg = state.cuda()
    got = call(_to_gpu(x), sg, None, rows.cuda())
    want = call(x, state, aux, rows)
    assert _rel(got, want) < 2e-5
    assert _rel(sg, state) < 2e-5


def test_recurrence_chunk_passes():
    """A step whose operands exceed the scratch limit runs in passes: the same
    results as two calls, each of which fits."""
    H, D, T = 160, 32, 9600
    g = torch.Generator(device="cuda").manual_seed(3)
    proj = torch.randn(T, 6 * H * D, generator=g, device="cuda",
                       dtype=torch.bfloat16)
    v = [proj[:, i * H * D:(i + 1) * H * D] for i in range(6)]
    par = [torch.randn(H * D, generator=g, device="cuda") for _ in range(3)]

    def run(parts):
        state = torch.zeros(1, H, D, D, device="cuda")
        outs = []
        for a, b in parts:
            rows = torch.tensor([[0, b - a, a, 0]], dtype=torch.int32,
                                device="cuda")
            outs.append(ops.delta_rule(*[t[a:b] for t in v], *par, state,
                                       rows, H, 1e-5, 0.6))
        return torch.cat(outs), state

    one, s1 = run([(0, T)])
    two, s2 = run([(0, T // 2), (T // 2, T)])
    assert torch.equal(one, two) and torch.equal(s1, s2)


@pytest.mark.parametrize("G,D,DV,chunk,window,softcap,learned", [
    (8, 128, 128, 64, 0, 0.0, False), (8, 64, 64, 0, 50, 0.0, True),
    (2, 128, 64, 0, 0, 0.0, True), (4, 64, 128, 40, 0, 9.0, True),
    (1, 64, 64, 33, 20, 0.0, False)])
def test_talk_attention_matrix_cores(G, D, DV, chunk, window, softcap,
                                     learned):
    """The 16-row head-mix kernel: portions that cross its row groups, rows
    of several sequences in one group, key counts around its 32-key tiles, a
    remainder of rows."""
    g = torch.Generator().manual_seed(14)
    H, bs, L = 32, 16, 150
    kc, vc, tables = _paged(L, G, D, DV, bs, torch.bfloat16, g, 3)
    ts, tp = [], []
    for s, a, b in ((0, 0, 35), (1, 60, 66), (2, 31, 34), (1, 95, 98),
                    (0, 127, 130), (2, 149, 150), (2, 0, 1)):
        ts += [s] * (b - a)
        tp += list(range(a, b))
    T = len(ts)
    q = torch.randn(T, H * D + 8, generator=g).to(torch.bfloat16)
    talk = torch.eye(H) + 0.3 * torch.randn(H, H, generator=g)
    sinks = torch.randn(H, generator=g) if learned else None
    ts = torch.tensor(ts, dtype=torch.int32)
    tp = torch.tensor(tp, dtype=torch.int32)
    want = reference.talk_attention(
        q[:, :H * D].float().reshape(T, H, D), kc.float(), vc.float(),
        tables, ts, tp, D ** -0.5, chunk, window, True, talk, 0, softcap,
        sinks)
    out = torch.full((T, H * DV + 4), 7.0, dtype=torch.bfloat16,
                     device="cuda")
    ops.talk_attention(
        q.cuda()[:, :H * D], kc.cuda(), vc.cuda(), tables.cuda(), ts.cuda(),
        tp.cuda(), D ** -0.5, H, chunk=chunk, window=window, sink=True,
        talk=talk.cuda(), softcap=softcap, variant=10,
        sink_vals=sinks.cuda() if learned else None, out=out[:, :H * DV])
    # fp32 up to the bf16 rounding of the result
    assert _rel(out[:, :H * DV].float().reshape(T, H, DV), want) < 3e-3
    assert (out[:, H * DV:] == 7.0).all()


@pytest.mark.parametrize("sink", [True, False])
@pytest.mark.parametrize("shape", ["up", "down", "steps"])
def test_talk_attention_scores_climb(shape, sink):
    """Scores that climb past the reference of the weights in nearly every half
    of a tile, once at its start, or in steps within first and second halves;
    rows of two sequences whose scores move by different amounts."""
    g = torch.Generator().manual_seed(19)
    H, G, D, DV, bs, L = 32, 8, 128, 128, 16, 170
    kc, vc, tables = _paged(L, G, D, DV, bs, torch.bfloat16, g, 2)
    pos = torch.arange(tables.shape[1] * bs).float()
    grow = {"up": 0.05 * pos, "down": 8.0 - 0.05 * pos,
            "steps": 2.0 * (pos // 21)}[shape]
    for s in range(2):
        # all heads' queries look along one direction, keys of sequence 1 less so
        f = grow * (1.0 if s == 0 else 0.4)
        for j in range(tables.shape[1]):
            kc[tables[s, j], :, :, 0] += f[j * bs:(j + 1) * bs].to(
                torch.bfloat16)
    ts = torch.tensor([0] * 25 + [1] * 12, dtype=torch.int32)
    tp = torch.tensor(list(range(140, 165)) + list(range(100, 112)),
                      dtype=torch.int32)
    T = len(ts)
    q = torch.randn(T, H, D, generator=g)
    q[:, :, 0] = 10.0 + q[:, :, 0].abs()
    q = q.to(torch.bfloat16)
    talk = torch.eye(H) + 0.1 * torch.randn(H, H, generator=g)
    want = reference.talk_attention(
        q.float(), kc.float(), vc.float(), tables, ts, tp, D ** -0.5, 0, 0,
        sink, talk)
    got = ops.talk_attention(
        q.cuda().view(T, H * D), kc.cuda(), vc.cuda(), tables.cuda(),
        ts.cuda(), tp.cuda(), D ** -0.5, H, sink=sink, talk=talk.cuda(),
        variant=10)
    # fp32 up to the bf16 rounding of the result; scores of up to 60 in sums of
    # 128 and 32 terms are 2e-5 off, and their weights with them
    assert _rel(got.float().cpu().reshape(T, H, DV), want) < 3e-3


@pytest.mark.parametrize("T,G,window", [(33, 8, 0), (45, 8, 0), (33, 8, 1500),
                                        (33, 8, 1550), (70, 8, 1500),
                                        (150, 8, 0), (320, 1, 0), (321, 1, 0)])
def test_window_attention_token_order(T, G, window):
    """Single tokens that workgroups take by their keys (a round of the CUs and
    one, two and a remainder, more than four, at the most and past it): every row
    is written, as a launch over few tokens (as they come) writes it."""
    g = torch.Generator().manual_seed(T)
    H, D, bs, nb = 2 * G, 64, 16, 300
    n = torch.tensor([1, 31, 32, 33, 500, 512, 513, 1000, 1000, 1600])
    pos = (n[torch.randint(0, 10, (T,), generator=g)] - 1).int()
    pos[T // 2] = 1599
    kc, vc = (torch.randn(nb, G, bs, D, generator=g).to(torch.bfloat16).cuda()
              for _ in range(2))
    tables = torch.randint(0, nb, (T, 100), generator=g).int().cuda()
    q = torch.randn(T, H * D, generator=g).to(torch.bfloat16).cuda()
    pos, seq = pos.cuda(), torch.arange(T, dtype=torch.int32).cuda()

    def run(a, b):
        return ops.talk_attention(
            q[a:b], kc, vc, tables, seq[a:b], pos[a:b], D ** -0.5, H,
            window=window, sink=True, keep_first=3 if window else 0, variant=3,
            splits=1).float()

    got, few = run(0, T), 256 // G
    # the same tiles in the same waves
    assert torch.equal(got, torch.cat([run(a, min(a + few, T))
                                       for a in range(0, T, few)]))


@pytest.mark.parametrize("grow", [0.03, 0.2, -0.1])
@pytest.mark.parametrize("softcap", [0.0, 50.0])
def test_window_attention_scores_climb(grow, softcap):
    """Scores that climb by less than the weights' reference waits for in a tile,
    by more than that in each, or fall from the first key on: as portions and as
    single tokens with one and several shares."""
    g = torch.Generator().manual_seed(29)
    H, G, D, bs, L = 8, 2, 64, 16, 330
    kc, vc, tables = _paged(L, G, D, D, bs, torch.bfloat16, g, 2)
    f = grow * torch.arange(tables.shape[1] * bs).float()
    for j in range(tables.shape[1]):
        kc[tables[0, j], :, :, 0] += f[j * bs:(j + 1) * bs].to(torch.bfloat16)
    ts = torch.tensor([0] * 40 + [1] * 12, dtype=torch.int32)
    tp = torch.tensor(list(range(280, 320)) + list(range(100, 112)),
                      dtype=torch.int32)
    T = len(ts)
    q = torch.randn(T, H, D, generator=g)
    q[:, :, 0] = 8.0 + q[:, :, 0].abs()
    q = q.to(torch.bfloat16)
    want = reference.talk_attention(
        q.float(), kc.float(), vc.float(), tables, ts, tp, D ** -0.5, 0, 250,
        True, None, softcap=softcap, keep_first=70)
    dev = [x.cuda() for x in (q.view(T, H * D), kc, vc, tables, ts, tp)]
    for kw in ({"variant": 0}, {"variant": 3},
               {"variant": 3, "splits": 3}):
        got = ops.talk_attention(*dev, D ** -0.5, H, window=250, sink=True,
                                 softcap=softcap, keep_first=70, **kw)
        # fp32 up to the bf16 rounding of the result; scores of up to 70 in sums
        # of 64 terms are 2e-5 off, and their weights with them
        assert _rel(got.float().cpu().reshape(T, H, D), want) < 3e-3, kw


@pytest.mark.parametrize("variant,splits,far", [
    (10, 0, 8), (11, 0, 4), (12, 1, 4), (12, 3, 4)])
@pytest.mark.parametrize("sink", [True, False])
def test_attention_largest_values(variant, splits, far, sink):
    """Values near the end of bf16's range at a key whose score lies nearly as
    far above the earlier ones as the weights' reference waits for (far powers of
    two): weights stay at most 1, so the sums do not overflow."""
    H, G, D, bs, L = 32, 8, 64, 16, 400
    kc = torch.zeros(L // bs, G, bs, D, dtype=torch.bfloat16)
    vc = torch.ones(L // bs, G, bs, D, dtype=torch.bfloat16)
    at = 389                                # no wave's first tile
    kc[at // bs, :, at % bs, 0] = 0.9 * far * math.log(2.0)
    vc[at // bs, :, at % bs, 5] = 1e38
    tables = torch.arange(L // bs, dtype=torch.int32).view(1, -1)
    tp = torch.arange(L - 8, L, dtype=torch.int32)
    ts = torch.zeros(8, dtype=torch.int32)
    q = torch.zeros(8, H, D, dtype=torch.bfloat16)
    q[:, :, 0] = 8.0
    talk = torch.eye(H) if variant == 10 else None
    want = reference.talk_attention(q.float(), kc.float(), vc.float(), tables,
                                    ts, tp, D ** -0.5, 0, 0, sink, talk)
    got = ops.talk_attention(
        q.view(8, H * D).cuda(), kc.cuda(), vc.cuda(), tables.cuda(), ts.cuda(),
        tp.cuda(), D ** -0.5, H, sink=sink, variant=variant, splits=splits,
        talk=talk.cuda() if talk is not None else None)
    # the bf16 rounding of the result, entry by entry
    err = (got.cpu().double().view(8, H, D) - want).abs() / want
    assert float(err.max()) < 5e-3


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,D", [(1, 32), (3, 32), (3, 64), (2, 128), (5, 96)])
def test_recurrence_readout_borders(H, D, dtype):
    """The read-out on 16-byte borders and off them (rows of the gate or of the
    result moved by one entry): several rows in a wave and several waves a row,
    rows of short segments between, before and behind those of chunks."""
    g = torch.Generator(device="cuda").manual_seed(23)
    rows = torch.tensor([[1, 40, 5, 2], [41, 3, 2, 0], [44, 17, 0, 1],
                         [0, 1, 4, 3], [61, 1, 9, 4]], dtype=torch.int32,
                        device="cuda")
    T, HD = 62, H * D
    v = [torch.randn(T, HD, generator=g, device="cuda").to(dtype)
         for _ in range(5)]
    par = [torch.randn(HD, generator=g, device="cuda") for _ in range(3)]
    gate = torch.randn(T, HD, generator=g, device="cuda").to(dtype)
    start = torch.randn(5, H, D, D, generator=g, device="cuda")

    def run(pitch, lead, out_lead):
        gp = torch.zeros(T, HD + pitch, dtype=dtype, device="cuda")
        gp[:, lead:lead + HD] = gate
        out = torch.full((T, HD + 16), 7.0, dtype=dtype, device="cuda")
        state = start.clone()
        ops.delta_rule(*v, gp[:, lead:lead + HD], *par, state, rows, H, 1e-5,
                       0.6, out=out[:, out_lead:out_lead + HD])
        assert (out[:, :out_lead] == 7.0).all()
        assert (out[:, out_lead + HD:] == 7.0).all()
        return out[:, out_lead:out_lead + HD].double(), state

    want, ws = run(16, 0, 0)
    for args in ((16, 1, 0), (17, 0, 0), (16, 0, 1)):
        got, st = run(*args)
        assert torch.equal(st, ws)
        # the squares' sum in another order: a step of fp32, or one of bf16 where
        # that crosses a border
        tol = 2e-6 if dtype == torch.float32 else 2 ** -7
        assert ((got - want).abs() <= tol * want.abs() + 1e-6).all()


def test_recurrence_softplus_range():
    """Step sizes of the state-space scan from the smallest to the largest argument,
    read from the state that one row of ones leaves: 2.3 steps of fp32 (as
    log1pf(expf()) has at most), and one more where the sum is rounded."""
    z = torch.cat([torch.linspace(-87, 100, 3000), torch.linspace(-4, 4, 1086),
                   torch.tensor([0.0, -0.0, 1e-30, -1e-30, 20.0, 2e4, 3e38,
                                 -3e38, float("inf"), float("-inf")])])
    H = z.numel()
    one = torch.ones(1, 1, device="cuda")
    state = torch.zeros(1, H, 1, 1, device="cuda")
    rows = torch.tensor([[0, 1, 0, 0]], dtype=torch.int32, device="cuda")
    zero = torch.zeros(H, device="cuda")
    ops.linear_scan("ssd", one, one, one.expand(1, H).contiguous(),
                    z.cuda()[None], zero[None], state, rows, H, 1, 1e-5,
                    p0=zero, p1=zero, p2=zero, normw=one[0])
    got, z = state.flatten().cpu().double(), z.double()
    want = z.clamp(min=0) + torch.log1p(torch.exp(-z.abs()))
    fin = torch.isfinite(want)
    assert torch.equal(got[~fin], want[~fin])
    got, want = got[fin], want[fin]
    # below 2^-126 a step no longer follows the number
    assert ((got - want).abs() <= 3.3 * 2 ** -24 * want + 2.0 ** -148).all()


@pytest.mark.parametrize("lens,chunk,window", [
    ([2040], 0, 0),                  # 128 blocks: as they come
    ([1500, 549], 512, 0),           # 129 by length, one of two sequences
    ([700] * 4, 0, 96),              # equal counts
    ([4099, 1000, 3], 64, 0)])       # 319, chunks of a few blocks
def test_talk_attention_block_order(lens, chunk, window):
    """Blocks of rows start by the keys they see: every row is written once,
    and as a launch over its own sequence alone writes it."""
    G, D, bs = 8, 64, 16
    T = sum(lens)
    g = torch.Generator(device="cuda").manual_seed(T)
    per = [-(-n // bs) for n in lens]
    kc, vc = (torch.randn(sum(per), G, bs, D, generator=g, device="cuda").to(
        torch.bfloat16) for _ in range(2))
    q = torch.randn(T, 32 * D, generator=g, device="cuda").to(torch.bfloat16)
    talk = torch.randn(32, 32, generator=g, device="cuda") * 0.2
    tables = torch.zeros(len(lens), max(per), dtype=torch.int32)
    for i, n in enumerate(per):
        tables[i, :n] = sum(per[:i]) + torch.arange(n)
    ts = torch.repeat_interleave(torch.arange(len(lens)), torch.tensor(lens))
    tp = torch.cat([torch.arange(n) for n in lens])
    tables, ts, tp = (x.int().cuda() for x in (tables, ts, tp))

    def run(a, b):
        out = torch.full((b - a, 32 * D), 7.0, device="cuda").to(
            torch.bfloat16)
        return ops.talk_attention(q[a:b], kc, vc, tables, ts[a:b], tp[a:b],
                                  D ** -0.5, 32, chunk=chunk, window=window,
                                  sink=True, talk=talk, out=out, variant=0)

    got, at = run(0, T), 0
    for n in lens:
        # bf16 rounding where blocks of 16 begin elsewhere: other tiles of keys
        assert _rel(got[at:at + n].float(), run(at, at + n).float()) < 3e-3
        at += n


@pytest.mark.parametrize("H,G,D,DV,window,keep,softcap,sink", [
    (8, 2, 128, 128, 0, 0, 0.0, None), (32, 4, 64, 64, 70, 3, 20.0, "zero"),
    (6, 2, 96, 40, 33, 64, 0.0, "heads"), (24, 1, 40, 128, 64, 66, 9.0, None),
    (200, 1, 8, 8, 100, 0, 0.0, "heads"), (5, 5, 128, 64, 1, 0, 0.0, None)])
def test_window_attention_kernels(H, G, D, DV, window, keep, softcap, sink):
    """Portions that cross the 128-row groups, rows of several sequences in
    one group, key counts around the 64- and 32-key tiles, kept keys before
    and inside the window, head counts that leave rows idle; as portions and
    as single tokens with one and several shares."""
    g = torch.Generator().manual_seed(15)
    bs, L = 16, 300
    kc, vc, tables = _paged(L, G, D, DV, bs, torch.bfloat16, g, 3)
    ts, tp = [], []
    for s, a, b in ((0, 0, 70), (1, 60, 66), (2, 31, 34), (1, 127, 130),
                    (0, 250, 300), (2, 299, 300), (2, 0, 1)):
        ts += [s] * (b - a)
        tp += list(range(a, b))
    T = len(ts)
    q = torch.randn(T, H * D + 8, generator=g).to(torch.bfloat16)
    sinks = torch.randn(H, generator=g) if sink == "heads" else None
    ts = torch.tensor(ts, dtype=torch.int32)
    tp = torch.tensor(tp, dtype=torch.int32)
    want = reference.talk_attention(
        q[:, :H * D].float().reshape(T, H, D), kc.float(), vc.float(),
        tables, ts, tp, D ** -0.5, 0, window, sink is not None, None, keep,
        softcap, sinks)
    for variant, splits in ((11, 0), (12, 1), (12, 0), (12, 5)):
        out = torch.full((T, H * DV + 4), 7.0, dtype=torch.bfloat16,
                         device="cuda")
        ops.talk_attention(
            q.cuda()[:, :H * D], kc.cuda(), vc.cuda(), tables.cuda(),
            ts.cuda(), tp.cuda(), D ** -0.5, H, window=window,
            keep_first=keep, sink=sink is not None, softcap=softcap,
            variant=variant, splits=splits, out=out[:, :H * DV],
            sink_vals=None if sinks is None else sinks.cuda())
        # fp32 up to the bf16 rounding of the result
        assert _rel(out[:, :H * DV].float().reshape(T, H, DV), want) < 3e-3
        assert (out[:, H * DV:] == 7.0).all()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("mode,H,D,DV", [
    ("gla", 2, 40, 72), ("gla", 1, 128, 33), ("ssd", 4, 64, 32),
    ("ssd", 2, 30, 40), ("mlstm", 2, 32, 31), ("mlstm", 1, 128, 64)])
def test_recurrence_chunk_runs(mode, H, D, DV, dtype):
    """Few heads and long segments: their chunks are walked in several runs
    at once. Runs with a remainder, runs that stay empty in shorter segments,
    fresh and continued states; a value that is no number reaches every later
    run of its segment and nothing else."""
    rows = _segs([700, 16, 401, 5, 90], [0, 3, 9, 0, 0])
    x, state, aux, call = _recurrence(mode, H, D, DV, rows, dtype)
    rows = torch.tensor(rows, dtype=torch.int32)
    sg = state.cuda()
    ag = aux.cuda() if aux is not None else None
    bad = _to_gpu(x)
    bad["v"][100] = float("nan")
    lost = call(bad, sg.clone(), None if ag is None else ag.clone(),
                rows.cuda())
    got = call(_to_gpu(x), sg, ag, rows.cuda())
    want = call(x, state, aux, rows)
    # 2^-24 a token over up to 700 of them, both sides; outputs rounded once
    assert _rel(got, want) < (2e-5 if dtype == torch.float32 else 6e-3)
    assert _rel(sg, state) < 5e-6
    if aux is not None:
        assert _rel(ag, aux) < 5e-6
    assert torch.equal(lost[:100], got[:100])
    assert torch.equal(lost[700:], got[700:])
    assert not torch.isfinite(lost[100:700]).all(1).any()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("W,n_out,top", [
    (64, 1, 1), (520, 3, 2), (4104, 5, 5), (2044, 17, 4), (4096, 70, 8)])
def test_moe_route_waves(W, n_out, top, dtype):
    """Both launch forms (up to 512 rows, more): the sums are made in the same
    order, so the same rows give the same bits; weights as the reference's."""
    g = torch.Generator().manual_seed(W)
    x = torch.randn(513, W, generator=g).to(dtype)
    rw = (torch.randn(n_out, W, generator=g) / W ** 0.5).to(dtype)
    many = ops.moe_route(x.cuda(), rw.cuda(), top)
    few = ops.moe_route(x[:512].cuda(), rw.cuda(), top)
    for a, b in zip(many, few):
        assert torch.equal(a[:512], b)
    want, sel, _ = reference.moe_route(x, rw, top, "softmax", True, None, 1.0,
                                       0.0)
    # logits are fp32 sums of W products; equal ones may change places
    assert (many[0].cpu() - want).abs().max() < 1e-4
    assert (many[1].cpu() == sel).float().mean() > 0.999


@pytest.mark.parametrize("softcap", [0.0, 20.0])
@pytest.mark.parametrize("low", [-math.inf, -3.4e38, -1e9, -1e4, 1e9, 3e38])
def test_window_attention_far_sinks(low, softcap):
    """Sinks far from every score, beside ordinary ones: a low one takes
    nothing, a high one everything, and neither costs the scores their
    digits."""
    g = torch.Generator().manual_seed(16)
    H, G, D, DV, bs, L = 8, 2, 64, 64, 16, 200
    kc, vc, tables = _paged(L, G, D, DV, bs, torch.bfloat16, g, 2)
    ts = torch.tensor([0] * 70 + [1] * 3, dtype=torch.int32)
    tp = torch.tensor(list(range(130, 200)) + [0, 1, 150], dtype=torch.int32)
    T = len(ts)
    q = torch.randn(T, H * D, generator=g).to(torch.bfloat16)
    sinks = torch.randn(H, generator=g)
    sinks[1::2] = low
    want = reference.talk_attention(
        q.float().reshape(T, H, D), kc.float(), vc.float(), tables, ts, tp,
        D ** -0.5, 0, 90, True, None, 3, softcap, sinks)
    for variant, splits in ((11, 0), (12, 1), (12, 3)):
        out = ops.talk_attention(
            q.cuda(), kc.cuda(), vc.cuda(), tables.cuda(), ts.cuda(),
            tp.cuda(), D ** -0.5, H, window=90, keep_first=3, sink=True,
            softcap=softcap, variant=variant, splits=splits,
            sink_vals=sinks.cuda()).float().cpu().reshape(T, H, DV)
        # fp32 up to the bf16 rounding of the result, head by head
        assert _rel(out[:, ::2], want[:, ::2]) < 3e-3
        if low > 0:
            assert (out[:, 1::2] == 0).all()
        else:
            assert _rel(out[:, 1::2], want[:, 1::2]) < 3e-3


@pytest.mark.parametrize("low", [-math.inf, -3.4e38, -1e9, -1e4, 1e9, 2.3e38,
                                 3.4e38])
@pytest.mark.parametrize("softcap", [0.0, 20.0])
def test_talk_attention_far_sinks(low, softcap):
    """Sinks far from every mixed score, beside ordinary ones: a low one takes
    nothing, a high one everything, up to the largest number."""
    g = torch.Generator().manual_seed(16)
    H, G, D, bs, L = 32, 8, 64, 16, 100
    kc, vc, tables = _paged(L, G, D, D, bs, torch.bfloat16, g, 2)
    ts = torch.tensor([0] * 30 + [1] * 3, dtype=torch.int32)
    tp = torch.tensor(list(range(60, 90)) + [0, 1, 95], dtype=torch.int32)
    T = len(ts)
    q = torch.randn(T, H * D, generator=g).to(torch.bfloat16)
    talk = torch.eye(H) + 0.1 * torch.randn(H, H, generator=g)
    sinks = torch.randn(H, generator=g)
    sinks[1::2] = low
    want = reference.talk_attention(
        q.float().reshape(T, H, D), kc.float(), vc.float(), tables, ts, tp,
        D ** -0.5, 0, 0, True, talk, 0, softcap, sinks)
    out = ops.talk_attention(
        q.cuda(), kc.cuda(), vc.cuda(), tables.cuda(), ts.cuda(), tp.cuda(),
        D ** -0.5, H, sink=True, softcap=softcap, talk=talk.cuda(), variant=10,
        sink_vals=sinks.cuda()).float().cpu().reshape(T, H, D)
    # fp32 up to the bf16 rounding of the result, head by head
    assert _rel(out[:, ::2], want[:, ::2]) < 3e-3
    if low > 0:
        assert (out[:, 1::2] == 0).all()
    else:
        assert _rel(out[:, 1::2], want[:, 1::2]) < 3e-3


@pytest.mark.parametrize("bad", [math.inf, -math.inf, math.nan])
@pytest.mark.parametrize("G,D,DV", [(8, 128, 128), (2, 64, 64)])
def test_talk_attention_value_no_number(G, D, DV, bad):
    """A cached value that is no finite number reaches the rows that see its
    key and no other: neither earlier rows of its sequence nor another
    sequence's in the same 16, to the last bit."""
    g = torch.Generator().manual_seed(17)
    H, bs, L = 32, 16, 120
    kc, vc, tables = _paged(L, G, D, DV, bs, torch.bfloat16, g, 2)
    # rows 0-5 sequence 0, 6-15 sequence 1, 16-20 sequence 0 again
    ts = torch.tensor([0] * 6 + [1] * 10 + [0] * 5, dtype=torch.int32)
    tp = torch.tensor(list(range(60, 66)) + list(range(90, 100))
                      + list(range(66, 71)), dtype=torch.int32)
    T = len(ts)
    q = torch.randn(T, H * D, generator=g).to(torch.bfloat16).cuda()
    talk = (torch.eye(H) + 0.3 * torch.randn(H, H, generator=g)).cuda()

    def run(v, variant):
        return ops.talk_attention(
            q, kc.cuda(), v.cuda(), tables.cuda(), ts.cuda(), tp.cuda(),
            D ** -0.5, H, window=40, sink=True, talk=talk,
            variant=variant).cpu().reshape(T, H, DV)

    clean = run(vc, 10)
    j, col = 94, 5                      # key 94 of sequence 1: rows 10-15
    broken = vc.clone()
    broken[tables[1, j // bs], 0, j % bs, col] = bad
    got = run(broken, 10)
    old = run(broken, 1)                # the general kernel
    sees = torch.zeros(T, H, DV, dtype=torch.bool)
    sees[10:16, :H // G, col] = True
    assert torch.equal(got[~sees], clean[~sees])
    for want in (math.inf, -math.inf):
        assert torch.equal(got == want, old == want)
    assert torch.equal(got.isnan(), old.isnan())
    assert not torch.isfinite(got[sees]).any()


@pytest.mark.parametrize("mode", ["general", "channel"])
def test_recurrence_chunk_long_keys(mode):
    """Keys whose squared norm leaves fp32's range: their unit vectors are
    zero in whole chunks as they are token by token."""
    segs = [(0, 20, 3, 0)]
    x, state, aux, call = _recurrence(mode, 2, 32, 32, segs, torch.float32)
    xg = _to_gpu(x)
    xg["k"][7] *= 1e20
    if mode == "channel":
        xg["q"][9] *= 1e20
    sg, st = state.cuda(), state.cuda()
    whole = call(xg, sg, None,
                 torch.tensor(segs, dtype=torch.int32).cuda())
    # the same rows in portions too short for a chunk
    parts = []
    for a in (0, 10):
        y = {k: v[a:a + 10] if v.shape[0] == 20 and v.dim() == 2 else v
             for k, v in xg.items()}
        parts.append(call(y, st, None, torch.tensor(
            [(0, 10, 3 + a, 0)], dtype=torch.int32).cuda()))
    assert torch.isfinite(whole).all()
    assert _rel(whole, torch.cat(parts)) < 2e-5
    assert _rel(sg, st) < 2e-5


@pytest.mark.parametrize("mode", RECURRENCES)
def test_recurrence_empty_segments(mode):
    """Segments without rows beside a long one: all of its rows are walked."""
    lens = [0, 60, 0, 0, 1] + [0] * 30
    rows = _segs(lens, [2] * len(lens))
    x, state, aux, call = _recurrence(mode, 2, 32, 32, rows, torch.float32)
    rows = torch.tensor(rows, dtype=torch.int32)
    sg = state.cuda()
    ag = aux.cuda() if aux is not None else None
    got = call(_to_gpu(x), sg, ag, rows.cuda())
    want = call(x, state, aux, rows)
    # fp32 sums of up to 60 tokens x 32 channels
    assert _rel(got, want) < 2e-5
    assert _rel(sg, state) < 2e-6
    if aux is not None:
        assert _rel(ag, aux) < 2e-6


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("mode", RECURRENCES)
@pytest.mark.parametrize("lens", [
    [33, 16, 0, 33, 70, 1, 16], [17 + i // 9 for i in range(32)],
    [16 + i % 3 for i in range(33)], [17] * 64,
    [1] * 31 + [20, 0, 40] + [7] * 29 + [33],
    [1, 0] + [16 + i % 3 for i in range(35)],
    [16 + i % 3 for i in range(65)]])
def test_recurrence_chunk_order(mode, lens, dtype):
    """Walks start by length, up to 32 segments of a chunk or more and 64 in
    all: equal lengths, empty and short segments among them, one segment more;
    values end with their segment, columns of the last workgroup beyond the
    head's."""
    rows = _segs(lens, [3 * (i % 2) for i in range(len(lens))])
    x, state, aux, call = _recurrence(mode, 2, 40, 40, rows, dtype)
    rows = torch.tensor(rows, dtype=torch.int32)
    sg = state.cuda()
    ag = aux.cuda() if aux is not None else None
    got = call(_to_gpu(x), sg, ag, rows.cuda())
    want = call(x, state, aux, rows)
    # fp32 sums of up to 70 tokens x 40 channels; two roundings to bf16
    assert _rel(got, want) < (2e-5 if dtype == torch.float32 else 6e-3)
    assert _rel(sg, state) < 2e-6
    if aux is not None:
        assert _rel(ag, aux) < 2e-6


@pytest.mark.parametrize("H,G,D,S,n", [
    (8, 8, 40, 70, 31),      # 128 rows a workgroup, of five sequences
    (8, 8, 64, 36, 31),      # 64 rows
    (16, 4, 64, 40, 13),     # 32 rows, of eight tokens
    (8, 8, 64, 2, 1100)])    # portions of many workgroups
def test_window_attention_row_groups(H, G, D, S, n):
    """Workgroups of 128, 64 and 32 rows that hold several sequences, one run
    from row 0 to 127, runs of single rows, runs that end on a group's last
    row."""
    g = torch.Generator().manual_seed(18)
    past = [5 * i % 40 for i in range(S)]
    kc, vc, tables = _paged(n + 40, G, D, D, 16, torch.bfloat16, g, S)
    ts = torch.cat([torch.full((n,), i) for i in range(S)]).int()
    tp = torch.cat([p + torch.arange(n) for p in past]).int()
    tp[130:137] = torch.tensor([9, 7, 5, 3, 1, 0, 2])  # rows on their own
    q = torch.randn(S * n, H * D, generator=g).to(torch.bfloat16).cuda()
    got, want = (ops.talk_attention(
        q, kc.cuda(), vc.cuda(), tables.cuda(), ts.cuda(), tp.cuda(),
        D ** -0.5, H, window=50, keep_first=2, sink=True, softcap=9.0,
        variant=v).float().reshape(-1, H, D) for v in (11, 1))
    # two roundings to bf16, row by row
    err = (got - want).norm(dim=-1) / want.norm(dim=-1)
    assert err.max().item() < 1e-2


@pytest.mark.parametrize("mode,T", [("general", 9700), ("mlstm", 20600)])
def test_recurrence_chunk_passes_of_segments(mode, T):
    """Passes that end inside a segment, between two and past the last: every
    segment as in a call of its own, bit for bit, and no more passes than the
    chunks need."""
    H, D = 160, 32
    g = torch.Generator(device="cuda").manual_seed(4)
    lens = [17, 3000, 1, 40, T - 3098, 16, 24]
    proj = torch.randn(T, 5 * H * D + 2 * H, generator=g, device="cuda",
                       dtype=torch.bfloat16)
    par = [torch.randn(H * D, generator=g, device="cuda") for _ in range(3)]
    first = torch.randn(len(lens), H, D, D, generator=g, device="cuda")
    norm = torch.rand(len(lens), H, D + 1, generator=g, device="cuda")
    q, k, v, zw, gate = (proj[:, i * H * D:(i + 1) * H * D]
                         for i in range(5))
    i, f = proj[:, 5 * H * D:5 * H * D + H], proj[:, 5 * H * D + H:]

    def run(rows, state, aux, a, b):
        rows = torch.tensor(rows, dtype=torch.int32, device="cuda")
        if mode == "general":
            return ops.delta_rule(q[a:b], k[a:b], v[a:b], zw[a:b], q[a:b],
                                  gate[a:b], *par, state, rows, H, 1e-5, 0.6)
        return ops.linear_scan(
            "mlstm", q[a:b], k[a:b], v[a:b], f[a:b], gate[a:b], state, rows,
            H, H, 1e-5, qscale=D ** -0.5, c0=5.0, wr=i[a:b], p0=par[0][:H],
            p1=par[1][:H], normw=par[2], aux=aux)

    starts = [sum(lens[:n]) for n in range(len(lens))]
    state, aux = first.clone(), norm.clone()
    got = run([(a, n, s % 2, s) for s, (a, n) in enumerate(zip(starts, lens))],
              state, aux, 0, T)
    one, aux1 = first.clone(), norm.clone()
    for s, (a, n) in enumerate(zip(starts, lens)):
        want = run([(0, n, s % 2, s)], one, aux1, a, a + n)
        assert torch.equal(got[a:a + n], want), s
    assert torch.equal(state, one) and torch.equal(aux, aux1)


def test_recurrence_chunk_many_segments():
    """Many segments whose operands exceed the scratch limit: a few passes, in
    less time than twice the rows of half as many take."""
    H, D, S, n = 32, 128, 256, 48
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(S * n, 6 * H * D, generator=g, device="cuda",
                    dtype=torch.bfloat16)
    v = [x[:, i * H * D:(i + 1) * H * D] for i in range(6)]
    par = [torch.randn(H * D, generator=g, device="cuda") for _ in range(3)]
    state = torch.zeros(S, H, D, D, device="cuda")

    def run(s):
        rows = torch.tensor([(i * n, n, 0, i) for i in range(s)],
                            dtype=torch.int32, device="cuda")
        part = [t[:s * n] for t in v]
        times = []
        for _ in range(4):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            out = ops.delta_rule(*part, *par, state, rows, H, 1e-5, 0.6)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return out, min(times)

    few, t_few = run(64)
    many, t_many = run(S)
    assert torch.equal(many[:64 * n], few)
    # four times the work; the passes by chunk number took 50 times as long
    assert t_many < 8 * t_few


@pytest.mark.parametrize("mode", RECURRENCES)
@pytest.mark.parametrize("lens", [
    (7,), (15, 1), (1, 1, 1), (40,), (17, 33), (40, 1, 2), (30, 9, 1, 16),
    (0, 5, 0), (0, 20)])
def test_recurrence_spans(mode, lens):
    """With the lengths known ahead: chunks alone, short segments alone token
    by token and through the sequential kernels, both, and empty segments."""
    rows = _segs(lens, [2 * i for i in range(len(lens))])
    x, state, aux, call = _recurrence(mode, 2, 32, 32, rows, torch.float32)
    spans = ops.segment_spans(rows)
    names = {"general": "delta_rule", "channel": "gated_delta"}
    op = getattr(ops, names.get(mode, "linear_scan"))
    rows = torch.tensor(rows, dtype=torch.int32)
    sg = state.cuda()
    ag = aux.cuda() if aux is not None else None
    with pytest.MonkeyPatch.context() as m:
        m.setattr(ops, op.__name__, lambda *a, **k: op(*a, **k, spans=spans))
        got = call(_to_gpu(x), sg, ag, rows.cuda())
    want = call(x, state, aux, rows)
    # fp32 sums of up to 40 tokens x 32 channels
    assert _rel(got, want) < 2e-5
    assert _rel(sg, state) < 2e-6
    if aux is not None:
        assert _rel(ag, aux) < 2e-6


def test_recurrence_spans_launches():
    """No launch for segments that are not there: what a batch of a few rows
    per sequence takes with and without its lengths."""
    S, n, H, D = 8, 12, 32, 128
    rows = [(i * n, n, 5, i) for i in range(S)]
    assert ops.segment_spans(rows) == (12, 12)
    assert ops.segment_spans([(0, 30, 0, 0), (30, 1, 4, 1)]) == (30, 1)
    assert ops.segment_spans([(0, 30, 0, 0), (30, 16, 4, 1)]) == (30, -1)
    forms = ops._segment_forms
    cells = H * D * D
    assert forms(96, S, cells, (12, 12)) == (False, True, False)
    assert forms(96, S, cells, (12, 12), "channel", H, D) == (
        False, True, False)
    assert forms(96, S, cells, (12, 12), "channel", 2 * H, 64) == (
        False, True, True)
    assert forms(8, 1, cells, (8, 8)) == (False, True, True)
    assert forms(8, 1, cells, (8, 8), "ssd", H, D) == (False, True, False)
    assert forms(8, 1, cells, (8, 8), "gla", 8, 256) == (False, True, False)
    assert forms(15, 1, cells, (15, 15), "mlstm", 8, 256) == (
        False, True, True)
    assert forms(64, S, cells, None) == (True, True, True)
    assert forms(64, 64, cells, None) == (False, True, True)
    assert forms(15, 1, cells, None) == (False, True, False)
    assert forms(512, 64, cells, (8, 8)) == (False, True, True)
    assert forms(46, 2, cells, (30, -1)) == (True, False, True)


@pytest.mark.parametrize("H,G,D,DV,chunk,window,keep,softcap", [
    (32, 8, 128, 128, 0, 90, 4, 0.0), (32, 8, 64, 64, 0, 0, 0, 30.0),
    (6, 2, 96, 80, 40, 0, 3, 0.0), (16, 1, 16, 4, 0, 33, 20, 0.0),
    (3, 3, 112, 128, 0, 0, 0, 0.0)])
@pytest.mark.parametrize("variant,splits", [(13, 1), (13, 3), (14, 1),
                                            (14, 4)])
def test_attention_fp32(H, G, D, DV, chunk, window, keep, softcap, variant,
                        splits):
    """The fp32 matrix-core kernel: portions that cross its row groups, rows of
    several sequences in one group, key counts around its 16-key tiles, shares
    without a key; a value that is no number and an infinite one, which only the
    rows that see them may show."""
    g = torch.Generator().manual_seed(14)
    bs, L = 16, 150
    kc, vc, tables = _paged(L, G, D, DV, bs, torch.float32, g, 3)
    ts, tp = [], []
    for s, a, b in ((0, 0, 35), (1, 60, 66), (2, 31, 34), (1, 95, 98),
                    (0, 127, 130), (2, 149, 150), (2, 0, 1)):
        ts += [s] * (b - a)
        tp += list(range(a, b))
    T = len(ts)
    q = torch.randn(T, H * D + 8, generator=g)
    sinks = torch.randn(H, generator=g)
    ts = torch.tensor(ts, dtype=torch.int32)
    tp = torch.tensor(tp, dtype=torch.int32)

    def run(kc, vc):
        want = reference.talk_attention(
            q[:, :H * D].reshape(T, H, D), kc, vc, tables, ts, tp, D ** -0.5,
            chunk, window, True, None, keep, softcap, sinks)
        out = torch.full((T, H * DV + 4), 7.0, device="cuda")
        ops.talk_attention(
            q.cuda()[:, :H * D], kc.cuda(), vc.cuda(), tables.cuda(),
            ts.cuda(), tp.cuda(), D ** -0.5, H, chunk=chunk, window=window,
            sink=True, softcap=softcap, variant=variant, keep_first=keep,
            sink_vals=sinks.cuda(), out=out[:, :H * DV], splits=splits)
        assert (out[:, H * DV:] == 7.0).all()
        return out[:, :H * DV].cpu().reshape(T, H, DV), want

    got, want = run(kc, vc)
    # sums of up to 150 and 128 roundings of 2^-24, scores of up to 5 before exp
    assert _rel(got, want) < 3e-6
    vc[tables[0, 128 // bs], 0, 128 % bs, 1] = float("nan")
    vc[tables[2, 32 // bs], 0, 32 % bs, 2] = float("inf")
    got, want = run(kc, vc)
    fin = torch.isfinite(want)
    assert torch.equal(fin, torch.isfinite(got))
    assert _rel(got[fin], want[fin]) < 3e-6


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("kw", [dict(window=100, keep_first=5),
                                dict(softcap=20.0), dict(chunk=70)])
def test_attention_fp32_wide(kw, splits, monkeypatch):
    """32 columns a wave, which 512 workgroups' rows and more take: rows of several
    sequences in a workgroup's eight, a last one of three, values that are no
    numbers and scores that are none."""
    lib = _Launches(ops._mx())
    monkeypatch.setattr(ops, "_mx", lambda: lib)
    g = torch.Generator(device="cuda").manual_seed(3)
    H, G, D, bs, T = 32, 8, 128, 16, 523
    kc, vc = (torch.randn(75, G, bs, D, generator=g, device="cuda")
              for _ in range(2))
    tables = torch.randperm(75, generator=g, device="cuda").int().view(3, 25)
    q = torch.randn(T, H * D, generator=g, device="cuda")
    ts, tp = [], []
    for s, a, b in ((0, 20, 291), (1, 0, 3), (2, 120, 366), (1, 3, 6)):
        ts += [s] * (b - a)
        tp += range(a, b)
    ts, tp = (torch.tensor(x, dtype=torch.int32, device="cuda")
              for x in (ts, tp))
    assert len(tp) == T
    for odd in (False, True):
        if odd:
            vc[tables[0, 200 // bs], 3, 200 % bs, 1] = float("nan")
            vc[tables[2, 300 // bs], 5, 300 % bs, 2] = float("inf")
            kc[tables[2, 310 // bs], 1, 310 % bs, 7] = float("nan")
        want, got = (ops.talk_attention(
            q, kc, vc, tables, ts, tp, D ** -0.5, H, sink=True, variant=v,
            splits=n, **kw) for v, n in ((2, 1), (13, splits)))
        name, args = lib.made[-1]
        assert name == "mx_attn_f32" and args[-4:-2] == (32, splits)
        fin = torch.isfinite(want)
        assert fin.all() != odd and torch.equal(fin, torch.isfinite(got))
        assert torch.equal(torch.isnan(want), torch.isnan(got))
        # sums of up to 366 and 128 roundings of 2^-24 on both sides
        assert _rel(got[fin], want[fin]) < 3e-6


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("G,D,DV,chunk,window,softcap,learned", [
    (8, 128, 128, 64, 0, 0.0, False), (8, 64, 64, 0, 50, 0.0, True),
    (2, 128, 64, 0, 0, 9.0, True), (1, 64, 128, 33, 20, 0.0, False)])
@pytest.mark.parametrize("splits", [1, 3])
def test_talk_attention_tokens(G, D, DV, chunk, window, softcap, learned,
                               splits, dtype):
    """The head-mix kernel of single tokens: key counts around its 16-key tiles
    and a workgroup's 64, shares without a key; a value that is no number and an
    infinite one, which only the heads and rows that see them may show."""
    g = torch.Generator().manual_seed(15)
    H, bs, L = 32, 16, 330
    kc, vc, tables = _paged(L, G, D, DV, bs, dtype, g, 3)
    tp = torch.tensor([0, 14, 15, 16, 62, 63, 64, 130, 191, 192, 193, 329],
                      dtype=torch.int32)
    T = len(tp)
    ts = (torch.arange(T) % 3).int()
    q = torch.randn(T, H * D + 8, generator=g).to(dtype)
    talk = torch.eye(H) + 0.2 * torch.randn(H, H, generator=g)
    sinks = torch.randn(H, generator=g) if learned else None

    def run(kc, vc):
        want = reference.talk_attention(
            q[:, :H * D].float().reshape(T, H, D), kc.float(), vc.float(),
            tables, ts, tp, D ** -0.5, chunk, window, True, talk, 0, softcap,
            sinks)
        out = torch.full((T, H * DV + 4), 7.0, dtype=dtype, device="cuda")
        ops.talk_attention(
            q.cuda()[:, :H * D], kc.cuda(), vc.cuda(), tables.cuda(),
            ts.cuda(), tp.cuda(), D ** -0.5, H, chunk=chunk, window=window,
            sink=True, talk=talk.cuda(), softcap=softcap, variant=15,
            sink_vals=sinks.cuda() if learned else None,
            out=out[:, :H * DV], splits=splits)
        assert (out[:, H * DV:] == 7.0).all()
        return out[:, :H * DV].cpu().reshape(T, H, DV), want

    got, want = run(kc, vc)
    # fp32 sums of up to 330 and 128 terms, or the bf16 rounding of the result
    bound = 3e-3 if dtype == torch.bfloat16 else 4e-6
    assert _rel(got, want) < bound
    vc[tables[1, 129 // bs], 0, 129 % bs, 1] = float("nan")
    vc[tables[2, 191 // bs], G - 1, 191 % bs, 2] = float("inf")
    got, want = run(kc, vc)
    fin = torch.isfinite(want)
    assert torch.equal(fin, torch.isfinite(got))
    assert _rel(got[fin], want[fin]) < bound


@pytest.mark.parametrize("G,D,DV,chunk,window,softcap,learned", [
    (8, 128, 128, 64, 0, 0.0, False), (8, 64, 64, 0, 50, 0.0, True),
    (2, 128, 64, 0, 0, 9.0, True), (1, 64, 128, 33, 20, 0.0, False)])
@pytest.mark.parametrize("splits", [1, 3])
def test_talk_attention_fp32_portions(G, D, DV, chunk, window, softcap,
                                      learned, splits):
    """The fp32 head-mix kernel of portions: rows that cross its groups of four,
    several sequences in one group, key counts around its 16-key tiles, shares
    without a key; a value that is no number and an infinite one, which only the
    heads and rows that see them may show."""
    g = torch.Generator().manual_seed(16)
    H, bs, L = 32, 16, 150
    kc, vc, tables = _paged(L, G, D, DV, bs, torch.float32, g, 3)
    ts, tp = [], []
    for s, a, b in ((0, 0, 35), (1, 60, 66), (2, 31, 34), (1, 95, 98),
                    (0, 127, 130), (2, 149, 150), (2, 0, 1)):
        ts += [s] * (b - a)
        tp += list(range(a, b))
    T = len(ts)
    q = torch.randn(T, H * D + 8, generator=g)
    talk = torch.eye(H) + 0.2 * torch.randn(H, H, generator=g)
    sinks = torch.randn(H, generator=g) if learned else None
    ts = torch.tensor(ts, dtype=torch.int32)
    tp = torch.tensor(tp, dtype=torch.int32)

    def run(kc, vc):
        want = reference.talk_attention(
            q[:, :H * D].reshape(T, H, D), kc, vc, tables, ts, tp, D ** -0.5,
            chunk, window, True, talk, 0, softcap, sinks)
        out = torch.full((T, H * DV + 4), 7.0, device="cuda")
        ops.talk_attention(
            q.cuda()[:, :H * D], kc.cuda(), vc.cuda(), tables.cuda(),
            ts.cuda(), tp.cuda(), D ** -0.5, H, chunk=chunk, window=window,
            sink=True, talk=talk.cuda(), softcap=softcap, variant=16,
            sink_vals=sinks.cuda() if learned else None,
            out=out[:, :H * DV], splits=splits)
        assert (out[:, H * DV:] == 7.0).all()
        return out[:, :H * DV].cpu().reshape(T, H, DV), want

    got, want = run(kc, vc)
    # fp32 sums of up to 150 and 128 terms
    assert _rel(got, want) < 4e-6
    vc[tables[0, 128 // bs], 0, 128 % bs, 1] = float("nan")
    vc[tables[2, 32 // bs], G - 1, 32 % bs, 2] = float("inf")
    got, want = run(kc, vc)
    fin = torch.isfinite(want)
    assert torch.equal(fin, torch.isfinite(got))
    assert _rel(got[fin], want[fin]) < 4e-6


@pytest.mark.parametrize("splits", [1, 2, 5, 16])
@pytest.mark.parametrize("D,DV,softcap", [(128, 128, 0.0), (64, 128, 9.0)])
def test_talk_attention_portion_shares(D, DV, softcap, splits):
    """The 16-row head-mix kernel with the keys of a block over several
    workgroups: shares of whole 32-key tiles, without a tile, without a key that
    a row of the block sees; a sink that counts once."""
    g = torch.Generator().manual_seed(18)
    H, G, bs, L, chunk = 32, 8, 16, 330, 200
    kc, vc, tables = _paged(L, G, D, DV, bs, torch.bfloat16, g, 2)
    ts, tp = [], []
    for s, a, b in ((0, 190, 215), (1, 0, 7), (1, 321, 330), (0, 31, 34)):
        ts += [s] * (b - a)
        tp += list(range(a, b))
    T = len(ts)
    q = torch.randn(T, H * D, generator=g).to(torch.bfloat16)
    talk = torch.eye(H) + 0.2 * torch.randn(H, H, generator=g)
    sinks = torch.randn(H, generator=g)
    ts, tp = (torch.tensor(x, dtype=torch.int32) for x in (ts, tp))
    want = reference.talk_attention(
        q.float().reshape(T, H, D), kc.float(), vc.float(), tables, ts, tp,
        D ** -0.5, chunk, 0, True, talk, 0, softcap, sinks)
    got = ops.talk_attention(
        *[x.cuda() for x in (q, kc, vc, tables, ts, tp)], D ** -0.5, H,
        chunk=chunk, sink=True, talk=talk.cuda(), softcap=softcap, variant=10,
        sink_vals=sinks.cuda(), splits=splits)
    # fp32 up to the bf16 rounding of the result
    assert _rel(got.float().cpu().reshape(T, H, DV), want) < 3e-3


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("lens,DV", [([64, 65], 32), ([63, 16], 30),
                                     ([1024, 17], 33), ([1025, 40], 32),
                                     ([2100, 1, 300], 64)])
def test_matrix_lstm_turns_of_waves(lens, DV, dtype):
    """The gates' running maximum over waves of 64 tokens, workgroups of 16 waves
    and several turns of them; outputs from rows on 16-byte borders and off them."""
    H, D = 3, 16
    segs = _segs(lens, [5, 0, 9][:len(lens)])
    x, state, aux, call = _recurrence("mlstm", H, D, DV, segs, dtype)
    # long stretches in which the maximum only decays, and steps up within them
    for k in ("a", "dec"):
        x[k][::] = (x[k].float() * 4 - (6 if k == "a" else 0)).to(dtype)
    rows = torch.tensor(segs, dtype=torch.int32)
    sr, ar = state.clone(), aux.clone()
    want = call({k: v.float() for k, v in x.items()}, sr, ar, rows)
    sg, ag = state.cuda(), aux.cuda()
    got = call(_to_gpu(x), sg, ag, rows.cuda())
    # sums over chunks of 16 or 32 rows; bf16 outputs are rounded
    assert _rel(got, want) < (4e-3 if dtype == torch.bfloat16 else 4e-6)
    assert _rel(sg, sr) < 4e-6 and _rel(ag, ar) < 4e-6
    assert _rel(ag[..., D], ar[..., D]) < 1e-6


@pytest.mark.parametrize("splits", [1, 2, 5, 16])
@pytest.mark.parametrize("H,G,D,DV,window,keep,softcap", [
    (32, 8, 128, 128, 700, 70, 0.0), (6, 2, 40, 72, 0, 0, 9.0)])
def test_window_attention_portion_shares(H, G, D, DV, window, keep, softcap,
                                         splits):
    """Portions whose keys several workgroups share: runs of some with shares and
    of one without in a workgroup's rows, a share of kept keys, shares without a
    key that a row sees, a sink that counts once also where share 0 has none."""
    g = torch.Generator().manual_seed(31)
    bs, L = 16, 1100
    kc, vc, tables = _paged(L, G, D, DV, bs, torch.bfloat16, g, 2)
    ts, tp = [], []
    for s, a, b in ((0, 940, 985), (1, 0, 7), (1, 1090, 1100), (0, 31, 34)):
        ts += [s] * (b - a)
        tp += list(range(a, b))
    T = len(ts)
    q = torch.randn(T, H * D, generator=g).to(torch.bfloat16)
    sinks = torch.randn(H, generator=g) * 2
    ts, tp = (torch.tensor(x, dtype=torch.int32) for x in (ts, tp))
    want = reference.talk_attention(
        q.float().reshape(T, H, D), kc.float(), vc.float(), tables, ts, tp,
        D ** -0.5, 0, window, True, None, keep, softcap, sinks)
    got = ops.talk_attention(
        *[x.cuda() for x in (q, kc, vc, tables, ts, tp)], D ** -0.5, H,
        window=window, sink=True, softcap=softcap, variant=11,
        keep_first=keep, sink_vals=sinks.cuda(), splits=splits)
    # fp32 up to the bf16 rounding of the result
    assert _rel(got.float().cpu().reshape(T, H, DV), want) < 3e-3


@pytest.mark.parametrize("talk", [False, True])
@pytest.mark.parametrize("longest", [0, 1, 130, 2000])
def test_attention_longest_hint(talk, longest):
    """Where the longest portion ends only plans the workgroups: unknown, too
    small, as it is, beyond the tables."""
    g = torch.Generator().manual_seed(33)
    H, G, D, bs, L = 32, 8, 64, 16, 1500
    kc, vc, tables = _paged(L, G, D, D, bs, torch.bfloat16, g, 2)
    ts = torch.tensor([0] * 40 + [1] * 17, dtype=torch.int32)
    tp = torch.cat([torch.arange(90, 130), torch.arange(17)]).int()
    T = len(ts)
    q = torch.randn(T, H * D, generator=g).to(torch.bfloat16)
    mix = torch.eye(H) + 0.2 * torch.randn(H, H, generator=g) if talk else None
    want = reference.talk_attention(
        q.float().reshape(T, H, D), kc.float(), vc.float(), tables, ts, tp,
        D ** -0.5, 0, 0, True, mix)
    got = ops.talk_attention(
        *[x.cuda() for x in (q, kc, vc, tables, ts, tp)], D ** -0.5, H,
        sink=True, talk=mix.cuda() if talk else None, longest=longest)
    # fp32 up to the bf16 rounding of the result
    assert _rel(got.float().cpu().reshape(T, H, D), want) < 3e-3


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("talk", [False, True])
@pytest.mark.parametrize("variant", [0, 3])
def test_attention_no_rows(dtype, talk, variant):
    """An empty batch has an empty result, whatever kernel would take it."""
    H, G, D, bs = 32, 8, 64, 16
    kc = torch.zeros(4, G, bs, D, dtype=dtype, device="cuda")
    none = torch.empty(0, dtype=torch.int32, device="cuda")
    mix = torch.eye(H, device="cuda") if talk else None
    out = ops.talk_attention(
        torch.empty(0, H * D, dtype=dtype, device="cuda"), kc, kc.clone(),
        torch.zeros(2, 4, dtype=torch.int32, device="cuda"), none, none,
        D ** -0.5, H, sink=True, talk=mix, variant=variant)
    assert out.shape == (0, H * D) and out.dtype == dtype


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("case", ["key", "key and value", "far", "query",
                                  "infinite key"])
@pytest.mark.parametrize("talk,variant,general", [
    (False, 13, 2), (False, 14, 4), (True, 16, 2), (True, 15, 4)])
def test_attention_fp32_scores_no_number(talk, variant, general, case, splits):
    """Scores that are no number, and values that are none behind a weight of
    zero, do what they do in the vector kernels: they hide their key in portions,
    whatever its value is, and reach the single tokens that see it."""
    g = torch.Generator().manual_seed(21)
    H, G, D, bs, L = 32, 8, 64, 16, 150
    kc, vc, tables = _paged(L, G, D, D, bs, torch.float32, g, 2)
    tp = torch.tensor([*range(40), *range(100, 150)], dtype=torch.int32)
    ts = torch.tensor([0] * 40 + [1] * 50, dtype=torch.int32)
    q = torch.randn(len(tp), H * D, generator=g)
    mix = torch.eye(H) + 0.2 * torch.randn(H, H, generator=g)
    nan, inf = float("nan"), float("inf")
    page, row = tables[1, 7], 9         # position 121 of sequence 1
    if case in ("key", "key and value"):
        kc[page, :, row, 3] = nan
    if case == "key and value":
        vc[page, :, row] = nan
    if case == "far":                   # exp of some -1000
        q, kc, mix = q.abs(), kc.abs(), torch.eye(H)
        kc[page, :, row] = -300.0
        vc[page, :, row, 5] = inf
    if case == "query":
        q[60, :D] = nan
    if case == "infinite key":
        q, mix = q.abs(), mix.abs()
        kc[page, :, row, 3] = -inf
        vc[page, :, row] = nan
    args = [x.cuda() for x in (q, kc, vc, tables, ts, tp)]
    want, got = (ops.talk_attention(
        *args, D ** -0.5, H, sink=True, talk=mix.cuda() if talk else None,
        variant=v, splits=s) for v, s in ((general, 1), (variant, splits)))
    assert torch.equal(torch.isnan(want), torch.isnan(got))
    fin = torch.isfinite(want)
    assert torch.equal(fin, torch.isfinite(got))
    # fp32 sums of up to 150 and 128 terms on both sides
    assert _rel(got[fin], want[fin]) < 4e-6


@pytest.mark.parametrize("talk,variant,dtype", [
    (False, 0, torch.bfloat16), (False, 11, torch.bfloat16),
    (True, 0, torch.bfloat16), (True, 10, torch.bfloat16),
    (False, 13, torch.float32), (False, 14, torch.float32),
    (True, 15, torch.float32), (True, 16, torch.float32)])
def test_attention_more_splits_than_records(talk, variant, dtype):
    """More shares than records are merged of are as many as that."""
    g = torch.Generator(device="cuda").manual_seed(1)
    H, G, D, bs, T = 32, 8, 64, 16, 9
    kc, vc = (torch.randn(40, G, bs, D, generator=g, device="cuda").to(dtype)
              for _ in range(2))
    tables = torch.randperm(40, generator=g, device="cuda").int()[None]
    q = torch.randn(T, H * D, generator=g, device="cuda").to(dtype)
    tp = torch.arange(T, dtype=torch.int32, device="cuda") + 610
    ts = torch.zeros_like(tp)
    mix = torch.eye(H, device="cuda") if talk else None
    a, b = (ops.talk_attention(q, kc, vc, tables, ts, tp, D ** -0.5, H,
                               talk=mix, variant=variant, splits=s)
            for s in (16, 40))
    assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,G,D,DV,talk,pitch", [
    (64, 1, 576, 512, False, 0),        # queries in a latent space
    (64, 1, 64, 64, False, 4),          # rows off 16-byte borders
    (24, 1, 128, 128, True, 0)])        # a mix over other than 32 heads
def test_attention_records_where_kernels_take_them(H, G, D, DV, talk, pitch,
                                                   dtype):
    """No memory for the records of a kernel that does not take the shape."""
    bs, T, blocks = 16, 20, 512
    kc = torch.zeros(blocks, G, bs, D, dtype=dtype, device="cuda")
    vc = kc if D == 576 else torch.zeros(blocks, G, bs, DV, dtype=dtype,
                                         device="cuda")
    tables = torch.arange(blocks, dtype=torch.int32, device="cuda")[None]
    q = torch.zeros(T, H * D + pitch // (2 if dtype == torch.float32 else 1),
                    dtype=dtype, device="cuda")[:, :H * D]
    tp = torch.arange(T, dtype=torch.int32, device="cuda") + 100
    out = torch.empty(T, H * DV, dtype=dtype, device="cuda")
    mix = torch.eye(H, device="cuda") if talk else None

    def run():
        ops.talk_attention(q, kc, vc, tables, torch.zeros_like(tp), tp, 0.1, H,
                           talk=mix, vdim=DV, out=out)

    run()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    run()
    # the zeros above and what the fall-back asks for are small
    assert torch.cuda.max_memory_allocated() - before < 1 << 16


@pytest.mark.parametrize("talk,dtype", [
    (False, torch.bfloat16), (True, torch.bfloat16),
    (False, torch.float32), (True, torch.float32)])
def test_attention_plan_is_of_the_keys(talk, dtype, monkeypatch):
    """A portion's shares do not depend on how many tables the call has; a hint
    takes the place of the tables' width. Where nobody counts the sequences, one
    alone has to gain by shares."""
    H, G, D, bs, T = 32, 8, 64, 16, 20
    lib = _Launches(ops._mx())
    monkeypatch.setattr(ops, "_mx", lambda: lib)
    kc, vc = (torch.zeros(160, G, bs, D, dtype=dtype, device="cuda")
              for _ in range(2))
    q = torch.zeros(T, H * D, dtype=dtype, device="cuda")
    tp = torch.arange(T, dtype=torch.int32, device="cuda") + 2400
    mix = torch.eye(H, device="cuda") if talk else None

    def shares(tables, longest=0, portions=1):
        ops.talk_attention(
            q, kc, vc, torch.arange(160, dtype=torch.int32,
                                    device="cuda").repeat(tables, 1),
            torch.zeros_like(tp), tp, D ** -0.5, H, talk=mix, longest=longest,
            portions=portions)
        return lib.shares()

    assert shares(1) > 2
    assert shares(1) == shares(4) == shares(5) == shares(100)
    assert shares(1, 2420) == shares(100, 2420) > 2
    assert shares(5, 100) < shares(5)
    assert shares(5, 100, 0) == shares(100, 100, 0) == shares(1, 100)
    assert shares(5, 0, 0) >= shares(5)


@pytest.mark.parametrize("talk", [False, True])
def test_attention_shares_of_far_scores(talk):
    """Scores around 65536 powers of two: shares of the keys meet as one walk adds
    them up. The scale makes no roundings of its own (it is half a power of two)."""
    g = torch.Generator().manual_seed(41)
    H, G, D, bs, L, T = 32, 8, 64, 16, 1024, 40
    kc, vc, tables = _paged(L, G, D, D, bs, torch.bfloat16, g, 1)
    q = torch.randn(T, H, D, generator=g)
    q[..., :32] = 64.0
    kc[..., :32] = 64.0
    kc[..., 32:] *= 0.25
    tp = torch.arange(L - T, L, dtype=torch.int32)
    args = [x.cuda() for x in (q.reshape(T, H * D).to(torch.bfloat16), kc, vc,
                               tables, torch.zeros_like(tp), tp)]
    mix = torch.eye(H, device="cuda") if talk else None
    one, more = (ops.talk_attention(
        *args, 0.5 * math.log(2), H, talk=mix, variant=10 if talk else 11,
        splits=s) for s in (1, 5))
    # the same weights but for roundings of 2^-24: at most one result in a hundred
    # goes to the next bf16 number, 2^-8 of it away
    assert _rel(more.float(), one.float()) < 0.1 * 2 ** -8
