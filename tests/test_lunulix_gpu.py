"""Lunulix on the GPU: every kernel against plain f64 references of the same
mechanism, then the model through the framework's step function, cache,
scheduler and graph against the oracle, in f32 and bf16."""

import lunulix_cases as C
import lunulix_oracle as O
import pytest
import torch

from quickstart_streaming_agents_amd.models.layers import RopeTable, StepPlan
from quickstart_streaming_agents_amd.ops import dispatch as D

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F32, BF = torch.float32, torch.bfloat16
BOTH = pytest.mark.parametrize("dtype", [F32, BF], ids=["f32", "bf16"])


def gen(seed):
    return torch.Generator().manual_seed(seed)


def rnd(g, *shape, dtype=F32, scale=1.0):
    return (torch.randn(*shape, generator=g) * scale).to(dtype)


def i32(*v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


def close(got, want, dtype):
    """Largest rms error of a row, relative to the rms of everything."""
    got, want = got.double().cpu(), want.double()
    rms = want.pow(2).mean().sqrt().clamp(min=1e-6)
    err = (got - want).pow(2).mean(-1).sqrt().max() / rms
    assert float(err) <= (2e-5 if dtype == F32 else 3e-2), float(err)


# ---- row kernels ------------------------------------------------------------

@BOTH
@pytest.mark.parametrize("W", [33, 100, 256, 4096, 8448])
@pytest.mark.parametrize("layer", [False, True])
def test_residual_norm_with_post_norm(W, layer, dtype):
    g = gen(W)
    T, V = 7, 11
    res, y = rnd(g, T, W), rnd(g, T, W, dtype=dtype)
    table, ids = rnd(g, V, W, dtype=dtype), torch.tensor([0, 10, 3, 3, 1, 9, 2])
    w, post = rnd(g, W, dtype=dtype), rnd(g, W, dtype=dtype)
    p = O.rms(y.double(), 1e-4, post.double())
    for init, full in ((True, True), (False, False)):
        r = res.to(DEV)
        out = D.residual_norm(
            r, y.to(DEV), w.to(DEV), None, 1e-4,
            table=table.to(DEV) if full else None,
            ids=ids.to(DEV) if full else None, init=init, layer=layer,
            post=post.to(DEV), tscale=3.5)
        x = p + (0 if init else res.double())
        if full:
            x = x + 3.5 * table.double()[ids]
        close(r, x, F32)
        c = x - x.mean(-1, keepdim=True) if layer else x
        close(out, O.rms(c, 1e-4, w.double()), dtype)
    # no weight: the stream itself
    r = res.to(DEV)
    out = D.residual_norm(r, y.to(DEV), None, None, 1e-4, post=post.to(DEV))
    close(r, res.double() + p, F32)
    close(out, res.double() + p, dtype)


@BOTH
@pytest.mark.parametrize("cols", [5, 24, 90, 264])
def test_gelu_units(cols, dtype):
    g = gen(1)
    x = rnd(g, 19, 2 * cols, dtype=dtype, scale=3.0)
    d = x.to(DEV)
    want = O.gelu_tanh(x[:, :cols].double())
    close(D.glu(d[:, :cols], d[:, cols:], "gelu"),
          want * x[:, cols:].double(), dtype)
    table = rnd(g, 13, 3 * cols, dtype=dtype)
    ids = torch.randint(0, 13, (19,), generator=g)
    for layer in range(3):
        got = D.glu_table(d[:, :cols], table.to(DEV), ids.to(DEV),
                          layer * cols)
        close(got, want * table[ids].double()[:, layer * cols:
                                              (layer + 1) * cols], dtype)


@BOTH
@pytest.mark.parametrize("parts,n", [(1, 36), (3, 7), (8, 512), (2, 1200),
                                     (5, 260)])
def test_part_norm(parts, n, dtype):
    g = gen(n)
    x, w = rnd(g, 9, parts * n, dtype=dtype), rnd(g, parts * n)
    out = torch.zeros(9, parts * n + 8, dtype=dtype, device=DEV)
    D.part_norm(x.to(DEV), w.to(DEV), out[:, 8:], parts, 1e-3)
    want = O.rms(x.double().view(9, parts, n), 1e-3).reshape(9, -1) * \
        w.double()
    close(out[:, 8:], want, dtype)
    assert not out[:, :8].any()


# ---- short convolutions -----------------------------------------------------

def _steps(lens, at):
    """Plan arrays of a step that brings lens[i] tokens from at[i] on for
    sequence i in slot 4 - i, all portions in one launch."""
    n = torch.tensor(lens)
    off = (n.cumsum(0) - n).tolist()
    item, t0 = [], []
    for i, m in enumerate(lens):
        for t in range(0, m, StepPlan.CONV_ROWS):
            item.append(i)
            t0.append(t)
    slots = [4 - i for i in range(len(lens))]
    return i32(*item), i32(*t0), i32(*off), i32(*at), i32(*lens), i32(*slots)


SCHEDULE = [[2, 17, 1, 40], [1, 1, 3, 2], [1, 1, 1, 1], [30, 2, 16, 1],
            [1, 1, 1, 1]]


@BOTH
@pytest.mark.parametrize("taps", [1, 2, 3, 4, 7])
@pytest.mark.parametrize("H,G,Dm,E,rot", [
    (3, 3, 13, 7, 6), (4, 2, 16, 24, 8), (6, 1, 32, 12, 32), (2, 1, 20, 8, 0)])
def test_conv_qkv(H, G, Dm, E, rot, taps, dtype):
    """Four sequences in steps of portions and single tokens: filters, turned
    q and k, pages, tails that start as garbage."""
    g = gen(taps * 100 + H)
    c = (H + G) * Dm + G * E
    total = [sum(s[i] for s in SCHEDULE) for i in range(4)]
    u = [rnd(g, t, c, dtype=dtype) for t in total]
    w = rnd(g, c, taps, dtype=BF)
    rope = RopeTable(rot, 500.0, DEV, C.STRETCH)
    rope.ensure(300)
    want = []
    for x in u:
        y = O.short_conv(x.double(), w.double())
        pos = torch.arange(len(x)).double()
        qk = O.rotate(y[:, :(H + G) * Dm].view(-1, H + G, Dm), pos, rot,
                      500.0, C.STRETCH)
        want.append((qk[:, :H].reshape(-1, H * Dm), qk[:, H:],
                     y[:, (H + G) * Dm:].view(-1, G, E)))
    tails = torch.full((6, taps - 1, c), float("nan"), dtype=dtype,
                       device=DEV)
    kc = torch.zeros(9, G, 64, Dm, dtype=dtype, device=DEV)
    vc = torch.zeros(9, G, 64, E, dtype=dtype, device=DEV)
    pages = [[7, 3], [1, 8], [0, 4], [5, 2]]
    filters = w.float().t().contiguous().to(DEV)
    at = [0] * 4
    for step in SCHEDULE:
        x = torch.cat([u[i][at[i]:at[i] + n] for i, n in enumerate(step)])
        pad = torch.zeros(len(x), c + (-c) % 8 + 8, dtype=dtype, device=DEV)
        pad[:, :c] = x.to(DEV)
        slots = [pages[i][p // 64] * 64 + p % 64 for i, n in enumerate(step)
                 for p in range(at[i], at[i] + n)]
        if all(n == 1 for n in step):
            conv = (None, None, None, i32(*[a + 1 for a in at]), None,
                    i32(4, 3, 2, 1))
        else:
            conv = _steps(step, at)
        q = D.conv_qkv(pad[:, :c], filters, tails, rope.cos, rope.sin, rot,
                       i32(*slots), kc, vc, H, *conv)
        close(q, torch.cat([want[i][0][at[i]:at[i] + n]
                            for i, n in enumerate(step)]), dtype)
        at = [a + n for a, n in zip(at, step)]
    for i, n in enumerate(total):
        p = torch.tensor([pages[i][t // 64] for t in range(n)])
        o = torch.arange(n) % 64
        close(kc.cpu()[p, :, o].reshape(n, -1), want[i][1].reshape(n, -1),
              dtype)
        close(vc.cpu()[p, :, o].reshape(n, -1), want[i][2].reshape(n, -1),
              dtype)
    # a row that is not in use leaves everything alone
    before = tails.clone(), kc.clone(), vc.clone()
    D.conv_qkv(pad[:4, :c], filters, tails, rope.cos, rope.sin, rot,
               i32(-1, -1, -1, -1), kc, vc, H, None, None, None,
               i32(0, 0, 0, 0), None, i32(-1, -1, -1, -1))
    for a, b in zip(before, (tails, kc, vc)):
        assert torch.equal(a.nan_to_num(9.0), b.nan_to_num(9.0))


@BOTH
@pytest.mark.parametrize("taps", [1, 2, 4, 6])
@pytest.mark.parametrize("c", [10, 36, 264])
def test_conv_silu(c, taps, dtype):
    g = gen(c)
    total = [sum(s[i] for s in SCHEDULE) for i in range(4)]
    u = [rnd(g, t, c, dtype=dtype) for t in total]
    w, b = rnd(g, c, taps, dtype=BF), rnd(g, c)
    want = [O.silu(O.short_conv(x.double(), w.double(), b.double()))
            for x in u]
    tails = torch.full((6, taps - 1, c), float("nan"), dtype=dtype,
                       device=DEV)
    at = [0] * 4
    for step in SCHEDULE:
        x = torch.cat([u[i][at[i]:at[i] + n] for i, n in enumerate(step)])
        conv = _steps(step, at) if max(step) > 1 else \
            (None, None, None, i32(*[a + 1 for a in at]), None,
             i32(4, 3, 2, 1))
        got = D.conv_silu(x.to(DEV), w.float().t().contiguous().to(DEV),
                          b.to(DEV), tails, *conv)
        close(got, torch.cat([want[i][at[i]:at[i] + n]
                              for i, n in enumerate(step)]), dtype)
        at = [a + n for a, n in zip(at, step)]


@BOTH
@pytest.mark.parametrize("taps", [2, 4, 5])
def test_conv_chunks_shared_or_whole(taps, dtype):
    """Few chunks are shared by several blocks, many are not: a step's portions
    together against one by one, which differ in nothing but that."""
    g = gen(taps)
    lens, at, c, H, G, Dm = [2200, 37, 1, 5], [0, 3, 64, 0], 96, 2, 1, 24
    x = rnd(g, sum(lens), c, dtype=dtype).to(DEV)
    w, b = rnd(g, taps, c).to(DEV), rnd(g, c).to(DEV)
    rope = RopeTable(8, 500.0, DEV, C.STRETCH)
    rope.ensure(2300)
    old = rnd(g, 6, taps - 1, c, dtype=dtype).to(DEV)
    pages = i32(*[i * 64 + p for i in range(40) for p in range(64)])

    def run(which):
        tails, tails2 = old.clone(), old.clone()
        kc = torch.zeros(40, G, 64, Dm, dtype=dtype, device=DEV)
        vc = torch.zeros(40, G, 64, Dm, dtype=dtype, device=DEV)
        out = []
        for ids in which:
            item, t0, off, start, n, slots = _steps([lens[i] for i in ids],
                                                    [at[i] for i in ids])
            slots = i32(*[4 - i for i in ids])
            rows = torch.cat([torch.arange(lens[i]) + sum(lens[:i])
                              for i in ids]).to(DEV)
            steps = item, t0, off, start, n, slots
            part = x[rows].contiguous()
            y = D.conv_silu(part, w, b, tails, *steps)
            q = D.conv_qkv(part, w, tails2, rope.cos, rope.sin, 8,
                           pages[rows].contiguous(), kc, vc, H, *steps)
            out.append(torch.cat([y, q], 1))
        return torch.cat(out), tails, tails2, kc, vc

    assert 2200 // 16 > 128
    for together, alone in zip(run([[0, 1, 2, 3]]), run([[0], [1], [2], [3]])):
        assert torch.equal(together, alone)
    # the long one in portions of few chunks, its tail carried from one to the next
    got = []
    tails = old.clone()
    for p in range(0, 2200, 320):
        m = min(320, 2200 - p)
        item, t0, off, _, n, _ = _steps([m], [p])
        got.append(D.conv_silu(x[p:p + m], w, b, tails, item, t0, off, i32(p),
                               n, i32(4)))
    y, t, *_ = run([[0]])
    assert torch.equal(torch.cat(got), y[:, :c])
    assert torch.equal(tails[4], t[4])


@BOTH
@pytest.mark.parametrize("taps", [1, 3, 4, 6])
def test_conv_one_by_one_or_ahead(taps, dtype):
    """More waves than the chip holds take their tokens one by one, a part of them
    several ahead, and so do portions of three and of four: not a bit differs."""
    g = gen(taps)
    H, G, Dm, rot, n = 40, 8, 24, 8, 8300
    c = (H + 2 * G) * Dm
    x, w, b = rnd(g, n, c, dtype=dtype).to(DEV), rnd(g, taps, c).to(DEV), \
        rnd(g, c).to(DEV)
    rope = RopeTable(rot, 500.0, DEV)
    rope.ensure(n)
    pages = torch.arange(n, dtype=torch.int32, device=DEV)

    def run(cuts):
        tails = [torch.zeros(5, taps - 1, c, dtype=dtype, device=DEV)
                 for _ in range(2)]
        kc = torch.zeros(n // 64 + 1, G, 64, Dm, dtype=dtype, device=DEV)
        vc, out, at = torch.zeros_like(kc), [], 0
        for m in cuts:
            item, t0, off, start, lens, slots = _steps([m], [at])
            steps = item, t0, off, start, lens, slots
            rows = slice(at, at + m)
            out.append(torch.cat([
                D.conv_qkv(x[rows], w, tails[0], rope.cos, rope.sin, rot,
                           pages[rows], kc, vc, H, *steps),
                D.conv_silu(x[rows], w, b, tails[1], *steps)], 1))
            at += m
        assert at == n
        return [torch.cat(out), kc, vc, *tails]

    # 168 threads' worth of channels: four waves for each 16 tokens
    assert n / 16 * 4 > 2048 > n / 32 * 4
    whole = run([n])
    for cuts in ([n // 2, n // 2], [n // 2 - 7, 3, 4, n // 2]):
        assert all(map(torch.equal, run(cuts), whole))


@pytest.mark.parametrize("taps", [1, 2, 3, 4, 6])
@pytest.mark.parametrize("n", [1, 3, 40, 1500])
def test_conv_qkv_turns_alike(taps, n):
    """The rotation's sums to the last bit in every form of a step: a token alone,
    few and many chunks, any filter.  A filter that passes its token through leaves
    f32 inputs as they are, and f64 holds a product of two of them whole."""
    g = gen(taps)
    H, G, Dm, rot = 2, 1, 24, 16
    c = (H + G) * Dm + G * Dm
    x, w = rnd(g, n, c), torch.zeros(taps, c)
    w[-1] = 1
    rope = RopeTable(rot, 500.0, DEV)
    rope.ensure(n)
    item, t0, off, start, lens, slots = _steps([n], [0])
    if n == 1:
        steps = (None, None, None, lens, None, slots)
    else:
        steps = (item, t0, off, start, lens, slots)
    kc = torch.zeros(n // 64 + 1, G, 64, Dm, device=DEV)
    vc = torch.zeros_like(kc)
    q = D.conv_qkv(x.to(DEV), w.to(DEV), torch.zeros(5, taps - 1, c, device=DEV),
                   rope.cos, rope.sin, rot, i32(*range(n)), kc, vc, H, *steps)
    cos, sin = (t[:n, None].cpu().double() for t in (rope.cos, rope.sin))
    qk = x[:, :(H + G) * Dm].view(n, H + G, Dm).double()
    a, b = qk[..., :rot // 2], qk[..., rot // 2:rot]
    want = torch.cat([a * cos - (b * sin).float().double(),
                      a * sin + (b * cos).float().double(), qk[..., rot:]], -1)
    assert torch.equal(q.cpu().view(n, H, Dm), want[:, :H].float())
    assert torch.equal(kc[:, 0].reshape(-1, Dm)[:n].cpu(), want[:, H].float())
    assert torch.equal(vc[:, 0].reshape(-1, Dm)[:n].cpu(), x[:, -Dm:])


# ---- attention --------------------------------------------------------------

@BOTH
@pytest.mark.parametrize("H,G,Dm,E", [
    (3, 3, 20, 18), (6, 2, 40, 72), (17, 1, 32, 32), (40, 2, 64, 48),
    (8, 2, 128, 128), (4, 1, 256, 136), (2, 1, 72, 256), (4, 4, 24, 16)])
def test_grouped_attention(H, G, Dm, E, dtype):
    """Rows and portions over a scattered page table whose other pages and
    unused places hold garbage; some rows single out one key at a page's edge,
    the first, or one far back."""
    g = gen(Dm + E)
    T, scale = 300, 0.8 * Dm ** -0.5
    q, k, v = (rnd(g, T, n, d, dtype=dtype)
               for n, d in ((H, Dm), (G, Dm), (G, E)))
    sink = rnd(g, H) + 1.0
    gate = rnd(g, T, H * E, dtype=dtype)
    for row, key in ((299, 0), (298, 63), (297, 64), (296, 127), (295, 128),
                     (130, 129), (200, 5), (64, 63), (65, 64)):
        for h in range(H):
            q[row, h] = (k[key, h // (H // G)].float() * 3).to(dtype)
    pages = [7, 2, 9, 4, 1]
    kc = torch.full((11, G, 64, Dm), 50.0, dtype=dtype)
    vc = torch.full((11, G, 64, E), float("nan"), dtype=dtype)
    for t in range(T):
        kc[pages[t // 64], :, t % 64] = k[t]
        vc[pages[t // 64], :, t % 64] = v[t]
    kc, vc = kc.to(DEV), vc.to(DEV)
    bt = torch.tensor([[0] * 5, pages], dtype=torch.int32, device=DEV)
    plain = O.sink_attention(q.double(), k.double(), v.double(), scale,
                             sink.double()).reshape(T, -1)
    want = plain * O.sigmoid(gate.double()) * 0.7
    qf = q.reshape(T, -1)
    some = [0, 1, 62, 63, 64, 65, 127, 128, 130, 190, 191, 200, 250, 295, 296,
            297, 298, 299]
    idx = torch.tensor(some)
    for row_item, table in ((i32(*[1] * len(some)), bt),
                            (None, bt[1:].repeat(len(some), 1))):
        out = torch.zeros(len(some), H * E + 8, dtype=dtype, device=DEV)
        D.gqa_rows(qf[idx].to(DEV), kc, vc, table, row_item,
                   (idx + 1).int().to(DEV), sink.to(DEV), gate[idx].to(DEV),
                   out[:, :H * E], H, scale, 0.7)
        close(out[:, :H * E], want[idx], dtype)
        assert not out[:, H * E:].any()
    # without sink and gate
    bare = O.sink_attention(q.double(), k.double(), v.double(), scale,
                            torch.full((H,), -1e30).double()).reshape(T, -1)
    out = torch.zeros(len(some), H * E, dtype=dtype, device=DEV)
    D.gqa_rows(qf[idx].to(DEV), kc, vc, bt, i32(*[1] * len(some)),
               (idx + 1).int().to(DEV), None, None, out, H, scale)
    close(out, bare[idx], dtype)
    # rows not in use come out as zero, without reading anything
    off = torch.ones(2, H * E, dtype=dtype, device=DEV)
    D.gqa_rows(qf[:2].to(DEV), kc, vc, bt, None, i32(0, 0), sink.to(DEV),
               None, off, H, scale)
    assert not off.any()
    if dtype != BF or not D.gqa_mfma_ok(Dm, E):
        return
    block = D.gqa_portion_rows(Dm, E)
    for start, n in ((0, 300), (63, 2), (64, 65), (130, 170), (200, 64),
                     (1, 128)):
        for s, gt, ref in ((sink.to(DEV), gate, want), (None, None, bare)):
            out = torch.empty(n, H * E, dtype=dtype, device=DEV)
            t0 = list(range(0, n, block))[::-1]
            D.gqa_portions(
                qf[start:start + n].to(DEV), kc, vc, bt[1:], s,
                None if gt is None else gt[start:start + n].to(DEV),
                i32(*[0] * len(t0)), i32(*t0), i32(0), i32(start), i32(n),
                out, H, scale, 0.7 if gt is not None else 1.0)
            close(out, ref[start:start + n], dtype)


@pytest.mark.parametrize("R,H,G,Dm,E", [
    (64, 16, 8, 128, 128), (129, 34, 2, 40, 24), (513, 1, 1, 256, 136)])
def test_grouped_attention_many_rows(R, H, G, Dm, E):
    """Enough rows for a block to finish its own: lengths without keys for
    some of its four shares, none at all, ends of pages."""
    g = gen(R)
    T, scale = 700, 0.8 * Dm ** -0.5
    q, k, v = (rnd(g, n, m, d, dtype=BF)
               for n, m, d in ((T, H, Dm), (T, G, Dm), (T, G, E)))
    sink, gate = rnd(g, H) + 1.0, rnd(g, T, H * E, dtype=BF)
    pages = [7, 2, 9, 4, 1, 3, 10, 0, 5, 8, 6]
    kc = torch.full((11, G, 64, Dm), 50.0, dtype=BF)
    vc = torch.full((11, G, 64, E), float("nan"), dtype=BF)
    for t in range(T):
        kc[pages[t // 64], :, t % 64] = k[t]
        vc[pages[t // 64], :, t % 64] = v[t]
    bt = torch.tensor([pages], dtype=torch.int32, device=DEV)
    edge = torch.tensor([0, 31, 63, 64, 127, 128, 191, 256, 699])
    idx = torch.cat([edge, torch.randint(0, T, (R - len(edge),),
                                         generator=g)])
    qf = q.reshape(T, -1)[idx].to(DEV)
    length = (idx + 1).int().to(DEV)
    length[-1] = 0
    for s, gt, mult in ((sink, gate, 0.7),
                        (torch.full((H,), -1e30), None, 1.0)):
        want = O.sink_attention(q.double(), k.double(), v.double(), scale,
                                s.double()).reshape(T, -1)
        if gt is not None:
            want = want * O.sigmoid(gt.double()) * mult
        want = want[idx]
        want[-1] = 0.0
        out = torch.zeros(R, H * E + 8, dtype=BF, device=DEV)
        D.gqa_rows(qf, kc.to(DEV), vc.to(DEV), bt, i32(*[0] * R), length,
                   s.to(DEV) if gt is not None else None,
                   None if gt is None else gt[idx].to(DEV),
                   out[:, :H * E], H, scale, mult)
        close(out[:, :H * E], want, BF)
        assert not out[:, H * E:].any()


@pytest.mark.parametrize("R", [3, 2100])
def test_grouped_attention_without_pages(R):
    """A table without columns: no row is in use."""
    H, Dm = 4, 32
    kc = torch.ones(1, 1, 64, Dm, dtype=BF, device=DEV)
    out = torch.ones(R, H * Dm, dtype=BF, device=DEV)
    D.gqa_rows(out.clone(), kc, kc, torch.zeros(R, 0, dtype=torch.int32,
                                                device=DEV), None,
               torch.zeros(R, dtype=torch.int32, device=DEV), None, None, out,
               H, 1.0)
    assert not out.any()


def test_portions_of_several_sequences():
    """One launch over portions of two sequences, rows behind each other."""
    g = gen(9)
    H, G, Dm, E, scale = 4, 2, 32, 48, 0.3
    lens, starts = [70, 150], [40, 0]
    bt = torch.tensor([[3, 0, 0], [5, 1, 4]], dtype=torch.int32)
    bt[0, 1] = 2
    kc = torch.zeros(6, G, 64, Dm, dtype=BF)
    vc = torch.zeros(6, G, 64, E, dtype=BF)
    q, want = [], []
    for i, (n, st) in enumerate(zip(lens, starts)):
        T = st + n
        qq, k, v = (rnd(g, T, m, d, dtype=BF)
                    for m, d in ((H, Dm), (G, Dm), (G, E)))
        for t in range(T):
            kc[bt[i, t // 64], :, t % 64] = k[t]
            vc[bt[i, t // 64], :, t % 64] = v[t]
        want.append(O.sink_attention(qq.double(), k.double(), v.double(),
                                     scale, torch.zeros(H).double())
                    [st:].reshape(n, -1))
        q.append(qq[st:].reshape(n, -1))
    block = D.gqa_portion_rows(Dm, E)
    item = [i for i, n in enumerate(lens) for _ in range(0, n, block)]
    t0 = [t for n in lens for t in range(0, n, block)]
    out = torch.empty(sum(lens), H * E, dtype=BF, device=DEV)
    D.gqa_portions(torch.cat(q).to(DEV), kc.to(DEV), vc.to(DEV), bt.to(DEV),
                   torch.zeros(H, device=DEV), None, i32(*item), i32(*t0),
                   i32(0, lens[0]), i32(*starts), i32(*lens), out, H, scale)
    close(out, torch.cat(want), BF)


@pytest.mark.parametrize("Dm,E", [(k, e) for k in (32, 64, 128, 248)
                                  for e in (24, 64, 128, 256)])
def test_portions_that_end_anywhere(Dm, E):
    """Every width of keys and values, portions of one to five pages whose
    waves end a page apart; slots that nobody has written hold NaN."""
    g = gen(Dm + E)
    H, G, scale = 4, 2, Dm ** -0.5
    items = [(a + d, n) for a in (0, 64, 128) for d, n in
             ((0, 1), (0, 64), (33, 32), (50, 31), (63, 2), (0, 129))]
    lens = [n for _, n in items]
    pages = [-(-(a + n) // 64) for a, n in items]
    bt = torch.zeros(len(items), max(pages), dtype=torch.int32)
    kc = torch.full((sum(pages), G, 64, Dm), float("nan"), dtype=BF)
    vc = torch.full((sum(pages), G, 64, E), float("nan"), dtype=BF)
    q, want, at = [], [], 0
    for i, (a, n) in enumerate(items):
        bt[i, :pages[i]] = torch.arange(at, at + pages[i])
        qq, k, v = (rnd(g, a + n, m, d, dtype=BF)
                    for m, d in ((H, Dm), (G, Dm), (G, E)))
        for p in range(pages[i]):
            rows = slice(p * 64, min(p * 64 + 64, a + n))
            kc[at + p, :, :rows.stop - rows.start] = k[rows].transpose(0, 1)
            vc[at + p, :, :rows.stop - rows.start] = v[rows].transpose(0, 1)
        at += pages[i]
        want.append(O.sink_attention(qq.double(), k.double(), v.double(),
                                     scale, torch.zeros(H).double())
                    [a:].reshape(n, -1))
        q.append(qq[a:].reshape(n, -1))
    block = D.gqa_portion_rows(Dm, E)
    item = [i for i, n in enumerate(lens) for _ in range(0, n, block)]
    t0 = [t for n in lens for t in range(0, n, block)]
    off = [sum(lens[:i]) for i in range(len(lens))]
    out = torch.empty(sum(lens), H * E, dtype=BF, device=DEV)
    D.gqa_portions(torch.cat(q).to(DEV), kc.to(DEV), vc.to(DEV), bt.to(DEV),
                   torch.zeros(H, device=DEV), None, i32(*item), i32(*t0),
                   i32(*off), i32(*[a for a, _ in items]), i32(*lens), out, H,
                   scale)
    close(out, torch.cat(want), BF)


# ---- state space ------------------------------------------------------------

SSD_SHAPES = [(3, 7, 13, 1), (4, 16, 8, 2), (2, 40, 48, 1), (6, 24, 32, 3),
              (4, 64, 128, 2), (2, 136, 96, 2), (1, 256, 256, 1),
              (5, 8, 64, 5)]


@BOTH
@pytest.mark.parametrize("H,P,N,G", SSD_SHAPES)
def test_ssd_kernels(H, P, N, G, dtype):
    """Portions (token loop and chunks) and single tokens, carrying the state
    from one to the next, with heads that forget at once and ones that
    hardly do."""
    g = gen(H * P)
    lens = [150, 64, 1, 2, 65, 3, 1]
    T, inner = sum(lens), H * P
    cx, zo = inner + 2 * G * N, 8
    dto = zo + inner + (-inner) % 8
    xbc = rnd(g, T, cx, dtype=dtype)
    u = rnd(g, T, dto + H + (-(dto + H)) % 8, dtype=dtype)
    A = torch.tensor([0.02, 8.0, 1.0, 300.0, 0.0, 0.3])[:H].contiguous()
    bias = torch.tensor([-1.0, 0.5, -3.0, 1.0, -2.0, 4.0])[:H].contiguous()
    skip = rnd(g, H)
    dt = O.softplus(u[:, dto:dto + H].double() + bias.double())
    z = u[:, zo:zo + inner].double()
    x = xbc[:, :inner].double().reshape(T, H, P)
    B, Cm = (xbc[:, inner + i * G * N:inner + (i + 1) * G * N].double()
             .reshape(T, G, N) for i in range(2))
    const = (A.to(DEV), bias.to(DEV), skip.to(DEV))
    for chunked in ([False, True] if dtype == BF else [False]):
        if chunked and not D.ssd_chunked_ok(H, N, P, G):
            continue
        state = torch.full((3, H, N, P), float("nan"), device=DEV)
        S, at = None, 0
        for n in lens:
            part = u[at:at + n].to(DEV), xbc[at:at + n].to(DEV)
            if n == 1:
                out = D.ssd_decode(part[0], zo, dto, part[1], *const, state,
                                   G, i32(2), i32(at + 1))
            else:
                out = torch.empty(n, inner, dtype=dtype, device=DEV)
                items = i32(2), i32(0), i32(at), i32(n)
                if chunked:
                    nch = -(-n // 64)
                    D.ssd_chunked(part[0], zo, dto, part[1], *const, state,
                                  G, *items, i32(0), i32(*[0] * nch),
                                  i32(*range(0, n, 64)), out)
                else:
                    D.ssd_seq(part[0], zo, dto, part[1], *const, state, G,
                              *items, out)
            r = slice(at, at + n)
            y, S = O.ssd_recurrence(x[r], B[r], Cm[r], dt[r], A.double(),
                                    skip.double(), S)
            close(out, y.reshape(n, inner) * O.silu(z[r]), dtype)
            # the state itself is f32-accurate on every path
            got = state[2].double().cpu()
            assert float((got - S).abs().max() /
                         S.pow(2).mean().sqrt()) < 3e-4
            at += n
    # rows not in use come out as zero and touch no state
    before = state.clone()
    out = D.ssd_decode(u[:2].to(DEV), zo, dto, xbc[:2].to(DEV), *const, state,
                       G, i32(-1, -1), i32(0, 0))
    assert not out.any()
    assert torch.equal(before.nan_to_num(9.0), state.nan_to_num(9.0))


# heads, vdim, state, groups, taps of either branch: 2, 4, 8 and 16 rows of state
# a thread, one and two waves of columns
STEPS = [(4, 64, 128, 4, 4, 4), (2, 64, 128, 1, 1, 3), (8, 64, 128, 2, 4, 4),
         (8, 64, 128, 1, 2, 1), (3, 128, 256, 3, 3, 2), (1, 256, 128, 1, 4, 4)]


@pytest.mark.parametrize("H,P,N,G,taps,qtaps", STEPS)
def test_ssd_step(H, P, N, G, taps, qtaps):
    """One launch for single tokens against the kernels it stands for: rows at
    their first tokens, later ones, and rows not in use."""
    g = gen(H * P + taps)
    B, QH, KG, Dm, E = 9, 6, 2, 40, 72
    inner, C = H * P, H * P + 2 * G * N
    qc = (QH + KG) * Dm + KG * E
    lens = [1, 2, 3, 4, 5, 900, 0, 64, 7]
    slots = [3, 0, 9, 2, 1, 8, 4, -1, 5]
    assert D.ssd_step_ok(H, N, P, G, G, taps)
    x = rnd(g, B, qc + 8, dtype=BF).to(DEV)
    u = rnd(g, B, C + inner + H + (-(C + inner + H)) % 8, dtype=BF).to(DEV)
    qw, w = (rnd(g, t, c).to(DEV) for t, c in ((qtaps, qc), (taps, C)))
    bias, skip, norm = (rnd(g, c).to(DEV) for c in (C, H, inner))
    A = torch.rand(H, generator=g).to(DEV) * 4
    db = rnd(g, H).to(DEV)
    rope = RopeTable(16, 1e4, DEV)
    rope.ensure(1000)

    def fresh():
        t = gen(7)
        return [rnd(t, *s, dtype=d).to(DEV) for s, d in (
            ((10, qtaps - 1, qc), BF), ((10, taps - 1, C), BF),
            ((10, H, N, P), F32), ((20, KG, 64, Dm), BF),
            ((20, KG, 64, E), BF))]

    def run(whole):
        qt, t, S, k, v = fresh()
        cache = i32(*[64 * i + 7 for i in range(B)])
        n, s = i32(*lens), i32(*slots)
        S[3] = float("nan")                      # row 0's, which is not read
        y = torch.full((B, inner + 8), 5., device=DEV, dtype=BF)
        a = (x[:, :qc], qw, qt, rope.cos, rope.sin, 16, cache, k, v, QH)
        if whole:
            q = D.ssd_step(*a, u, w, bias, t, A, db, skip, S, G, norm, 1e-4,
                           y[:, 8:], s, n)
        else:
            conv = (None, None, None, n, None, s)
            q = D.conv_qkv(*a, *conv)
            o = D.ssd_decode(u, 0, inner + C, D.conv_silu(
                u[:, inner:inner + C], w, bias, t, *conv), A, db, skip, S, G,
                s, n)
            D.part_norm(o, norm, y[:, 8:], G, 1e-4)
        live = torch.tensor([i for i in range(B) if lens[i] and slots[i] >= 0])
        return [q[live], y, qt, t, S.nan_to_num(9.), k, v]

    got, want = run(True), run(False)
    for i in (0, 2, 3, 5, 6):                    # copies of one code
        assert torch.equal(got[i], want[i]), i
    # f32 in the same order but for the read-out's sums over N
    assert float((got[4] - want[4]).abs().max()) <= 1e-5 * float(
        want[4].abs().max())
    close(got[1][:, 8:], want[1][:, 8:].cpu(), BF)
    assert not got[1][[6, 7], 8:].any() and (got[1][:, :8] == 5).all()


@pytest.mark.parametrize("case", [(3, 13, 7, 1, 1, 4), (8, 128, 64, 2, 4, 4),
                                  (8, 128, 64, 2, 2, 5), (6, 128, 64, 2, 2, 4),
                                  (16, 128, 64, 1, 1, 4)])
def test_ssd_step_refuses(case):
    """Norm parts that are not the groups, long filters, columns and states
    that threads do not divide: the general kernels take those."""
    assert not D.ssd_step_ok(*case)


def test_ssd_step_refuses_host_operands():
    """Each operand whose memory is the host's is an error, not a launch."""
    g, B, H, N, P, G, QH, KG, Dm, E = gen(1), 3, 4, 64, 128, 4, 2, 1, 8, 8
    inner, C, qc = H * P, H * P + 2 * G * N, (QH + KG) * Dm + KG * E
    rope = RopeTable(8, 1e4, DEV)
    rope.ensure(10)
    args = [rnd(g, B, qc, dtype=BF).to(DEV), rnd(g, 4, qc).to(DEV),
            rnd(g, B, 3, qc, dtype=BF).to(DEV), rope.cos, rope.sin, 8,
            i32(0, 64, 128), rnd(g, 3, KG, 64, Dm, dtype=BF).to(DEV),
            rnd(g, 3, KG, 64, E, dtype=BF).to(DEV), QH,
            rnd(g, B, inner + C + H, dtype=BF).to(DEV),
            rnd(g, 4, C).to(DEV), rnd(g, C).to(DEV),
            rnd(g, B, 3, C, dtype=BF).to(DEV), rnd(g, H).to(DEV),
            rnd(g, H).to(DEV), rnd(g, H).to(DEV), rnd(g, B, H, N, P).to(DEV), G,
            rnd(g, inner).to(DEV), 1e-5,
            torch.zeros(B, inner, device=DEV, dtype=BF), i32(0, 1, 2),
            i32(1, 5, 9)]
    assert torch.isfinite(D.ssd_step(*args)).all()
    for i, t in enumerate(args):
        if isinstance(t, torch.Tensor):
            with pytest.raises(RuntimeError):
                D.lm_ext().ssd_step(*args[:i], t.cpu(), *args[i + 1:])


# ---- the model through the framework ----------------------------------------

@pytest.fixture(scope="module")
def cases():
    return {(n, t): C.Case(n, DEV, t) for n in C.CONFIGS for t in (F32, BF)}


NAMES = pytest.mark.parametrize("name", list(C.CONFIGS))


def test_steps_in_one_launch(cases):
    """Which models' single tokens take the one launch: those of "groups", stored
    in bf16, in every layer."""
    for (name, dtype), case in cases.items():
        whole = [L.mixer.whole for L in case.model.layers]
        assert all(whole) if (name, dtype) == ("groups", BF) else not any(whole)


@BOTH
@NAMES
def test_residual_after_every_layer(cases, name, dtype):
    case = cases[name, dtype]
    toks = case.tokens(90)
    kv = case.model.new_kv_cache(2, 1)
    kv.allocate(0, 90)
    trail = []
    case.model.forward_prefill_batch(
        [(torch.tensor(toks, device=DEV), 0, 0)], kv, trail=trail)
    want = O.forward(case.raw, case.weights, toks)[1]
    assert len(trail) == len(want)
    for a, b in zip(trail, want):
        err = (a.double().cpu() - b).pow(2).mean().sqrt() / \
            b.pow(2).mean().sqrt()
        assert float(err) < (2e-5 if dtype == F32 else 2e-2)


@BOTH
@NAMES
@pytest.mark.parametrize("cuts", list(C.CUTS))
def test_cuts(cases, name, cuts, dtype):
    C.scenario_cuts(cases[name, dtype], 150, cuts)


@BOTH
@NAMES
def test_mixed_batches(cases, name, dtype):
    for seed in range(2):
        C.scenario_mixed(cases[name, dtype], seed)


@BOTH
@NAMES
def test_slot_and_page_reuse(cases, name, dtype):
    C.scenario_reuse(cases[name, dtype])


@BOTH
@pytest.mark.parametrize("spot,n", [(0, 200), (63, 150), (64, 200)])
@pytest.mark.parametrize("cuts", [
    lambda n: [n], lambda n: [n - 12] + [1] * 12,
    lambda n: C.portions(n, [2, 37])], ids=["prompt", "decoded", "portions"])
def test_far_keys(spot, n, cuts, dtype):
    C.scenario_far_key(spot, n, DEV, dtype, cuts)


@BOTH
def test_long_prompt_and_long_decoding(cases, dtype):
    case = cases["ones", dtype]
    C.scenario_cuts(case, 1000, "whole")
    C.scenario_cuts(case, 700, "decoded tail")


@BOTH
@pytest.mark.parametrize("chunk", [None, 24])
@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("name", ["odd", "tiles", "groups"])
def test_generation(cases, name, chunk, graph, dtype):
    C.scenario_generate(cases[name, dtype], use_graph=graph,
                        chunk_tokens=chunk)


@BOTH
@pytest.mark.parametrize("name", ["tiles", "groups"])
def test_graph_replays_match_eager_steps(cases, name, dtype):
    """Captured decode runs, several in a row with eager work between them,
    against eager decoding of the same prompts."""
    case = cases[name, dtype]
    prompts = [case.tokens(n, seed=n) for n in (70, 3, 129)]
    eng = case.engine(1024)
    ref = case.engine(1024)
    ref.use_graph = False
    for again in range(3):
        a = eng.generate_batch(prompts, [20, 20, 20])
        assert eng.use_graph and not eng._graph_failed
        b = ref.generate_batch(prompts, [20, 20, 20])
        if dtype == F32:
            assert a == b
        for p, o in zip(prompts, a):
            C.greedy_check(case, p, o)
        torch.zeros(64, 1024, device=DEV).normal_().sum().item()


@BOTH
@pytest.mark.parametrize("name", ["tiles", "groups"])
def test_conversations_reuse_the_snapshot(cases, name, dtype):
    C.scenario_conversation(cases[name, dtype])


def test_preset_on_engine():
    from quickstart_streaming_agents_amd.models import build_model
    from quickstart_streaming_agents_amd.models.serve import Engine, EngineLLM
    llm = EngineLLM(Engine(build_model("tiny-lunulix", device=DEV),
                           max_batch=4, max_seq_len=512))
    out = llm(["price of boots?", "hello"], [8, 8], ["a", "b"])
    assert len(out) == 2
    llm.release_all()
    assert llm.engine.kv.free_slots == llm.engine.kv.n_slots


@pytest.mark.parametrize("R,H,G,Dm,E,pages", [
    (129, 8, 8, 64, 64, 3), (129, 8, 8, 64, 64, 4),    # 1032 tiles
    (257, 16, 8, 128, 128, 7), (257, 16, 8, 128, 128, 8),
    (513, 2, 1, 200, 24, 7), (513, 2, 1, 200, 24, 8),
    (801, 2, 1, 24, 136, 8), (64, 8, 8, 200, 200, 1)])
def test_grouped_attention_forms(R, H, G, Dm, E, pages):
    """Both sides of the rule between shares and a block's own rows, which
    looks at rows, head sizes and the table's width: rows without keys, of one
    key and of all."""
    g = gen(R + pages)
    kc, vc = rnd(g, pages, G, 64, Dm, dtype=BF), rnd(g, pages, G, 64, E,
                                                     dtype=BF)
    q = rnd(g, R, H * Dm, dtype=BF)
    n = torch.randint(0, pages * 64 + 1, (R,), generator=g)
    n[:3] = torch.tensor([0, 1, pages * 64])
    bt = torch.randperm(pages, generator=g).int().repeat(R, 1)
    out = torch.empty(R, H * E, dtype=BF, device=DEV)
    D.gqa_rows(q.to(DEV), kc.to(DEV), vc.to(DEV), bt.to(DEV), None,
               n.int().to(DEV), None, None, out, H, Dm ** -0.5, 1.0)
    k, v = (t[bt[0].long()].transpose(0, 1).reshape(G, pages * 64, -1)
            .double().repeat_interleave(H // G, 0) for t in (kc, vc))
    s = torch.einsum("rhd,hjd->rhj", q.double().view(R, H, Dm), k) * Dm ** -0.5
    s = s.masked_fill(torch.arange(pages * 64) >= n[:, None, None],
                      float("-inf"))
    want = torch.einsum("rhj,hje->rhe", s.softmax(-1).nan_to_num(0.0), v)
    close(out, want.reshape(R, -1), BF)


# fewer than 512 tiles: up to 8 pages, 129 tiles to 16, 192 tiles
@pytest.mark.parametrize("R,H,G,Dm,E,pages", [
    (4, 16, 8, 128, 128, 8), (4, 16, 8, 128, 128, 9), (16, 8, 8, 64, 64, 16),
    (43, 3, 3, 40, 72, 16), (43, 3, 3, 40, 72, 17), (24, 8, 8, 128, 128, 17),
    (5, 2, 1, 136, 128, 3)])
def test_grouped_attention_few_rows(R, H, G, Dm, E, pages):
    test_grouped_attention_forms(R, H, G, Dm, E, pages)


# ---- projections of larger decode batches -----------------------------------

@pytest.mark.parametrize("M", [1, 33, 48, 49, 65, 97, 128, 129, 192])
@pytest.mark.parametrize("N,K", [(16, 64), (144, 192), (2048, 8192)])
def test_rows_gemm(M, N, K):
    """Ends of row tiles, column blocks and shares of K; rows of a slice.  An
    f32 sum of K products and a rounding to bf16."""
    from quickstart_streaming_agents_amd.ops import lm_ext
    g = gen(M + N)
    x = rnd(g, M, K + 24, dtype=BF)[:, 8:K + 8].to(DEV)
    w = rnd(g, N, K, dtype=BF).to(DEV)
    got = lm_ext().rows_gemm(x, w).double()
    a, b = x.double(), w.double()
    bound = 2.0 ** -8 * (a @ b.T).abs() + K * 2.0 ** -24 * (a.abs() @ b.abs().T)
    assert ((got - a @ b.T).abs() <= bound).all()


@pytest.mark.parametrize("M", [33, 192])
@pytest.mark.parametrize("N,K", [(1280, 2112), (2576, 4160)])
def test_rows_gemm_uneven_shares(M, N, K):
    """Columns that divide the chip with a remainder, shares of unlike length
    (33 steps of K in 25, 65 in 12)."""
    test_rows_gemm(M, N, K)


# sizes that the rule gives to every tile, with ends inside tiles and shares
ROWS_SIZES = [(65, 32, 128), (33, 10768, 128), (40, 2048, 1024),
              (64, 28688, 512), (257, 6160, 1088), (100, 4112, 4096),
              (330, 10096, 128), (1000, 3104, 1088), (130, 2032, 8256),
              (191, 4112, 4032), (330, 12304, 192), (700, 9696, 832),
              (300, 16416, 576), (700, 8256, 64), (2100, 4112, 576),
              (385, 16400, 704), (1500, 6176, 1024), (1000, 8880, 576),
              (1700, 8208, 256), (167, 16384, 2048), (70, 10240, 512),
              (1159, 9376, 128), (1283, 8128, 1600)]


def stale(*shape):
    """Leaves NaN where the next tensor of this size will be."""
    torch.full(shape, float("nan"), dtype=BF, device=DEV)


@pytest.mark.parametrize("M,N,K", ROWS_SIZES)
def test_rows_gemm_tiles(M, N, K):
    x, w = (rnd(gen(M + N), n, K, dtype=BF).to(DEV) for n in (M, N))
    stale(M, N)
    got = D.rows_linear(x, w).double()
    a, b = x.double(), w.double()
    bound = 2.0 ** -8 * (a @ b.T).abs() + K * 2.0 ** -24 * (a.abs() @ b.abs().T)
    assert ((got - a @ b.T).abs() <= bound).all()


@pytest.mark.parametrize("act", ["silu", "gelu", "silu of sums"])
@pytest.mark.parametrize("M,N,K", ROWS_SIZES)
def test_rows_glu(M, N, K, act):
    """Gate and up are rounded to bf16 (but for sums) after the product's f32
    error, e in all, and both activations have a slope of at most 1.13; __expf and the division
    are good to some 2^-20, the result is rounded to bf16."""
    N = N // 32 * 32
    g = gen(M + N)
    x = rnd(g, M, K + 24, dtype=BF)[:, 8:K + 8].to(DEV)
    w = rnd(g, N, K, dtype=BF, scale=K ** -0.5).to(DEV)
    stale(M, N // 2)
    sums = act == "silu of sums"
    act = act.split()[0]
    got = D.glu_linear(x, w, act, not sums).double()
    a, b = x.double(), w.double()
    e = K * 2.0 ** -24 * (a.abs() @ b.abs().T) + 2.0 ** -20 \
        + (0.0 if sums else 2.0 ** -8) * (a @ b.T).abs()
    (p, q), (ep, eq) = (a @ b.T).chunk(2, 1), e.chunk(2, 1)
    f = torch.nn.functional.silu(p) if act == "silu" else \
        torch.nn.functional.gelu(p, approximate="tanh")
    bound = (2.0 ** -8 + 2.0 ** -18) * (f * q).abs() + 1.13 * ep * q.abs() \
        + (f.abs() + ep) * eq
    assert ((got - f * q).abs() <= bound).all()


def test_rows_gemm_sizes_reach_every_tile():
    from quickstart_streaming_agents_amd.ops import lm_ext
    plain = {lm_ext().rows_gemm_plan(*s, False)[0] for s in ROWS_SIZES}
    assert plain == set(range(14))
    gated = {lm_ext().rows_gemm_plan(m, n // 32 * 32, k, True)[0]
             for m, n, k in ROWS_SIZES}
    assert gated == set(range(14)) - {0, 9}       # no pairs of column tiles


@pytest.mark.parametrize("M", [1, 3, 4, 7, 8, 16, 17, 32, 33])
@pytest.mark.parametrize("N,K", [(512, 1536), (512, 1024), (512, 512),
                                 (5632, 512), (512, 4096)])
def test_linear_by_rows(M, N, K):
    """Either side of the rows at which a product leaves the packed stream."""
    from quickstart_streaming_agents_amd.models.layers import Linear
    lin = Linear(rnd(gen(N + K), N, K, dtype=BF).to(DEV))
    x = rnd(gen(M), M, K, dtype=BF).to(DEV)
    a, b = x.double(), lin.w.double()
    bound = 2.0 ** -8 * (a @ b.T).abs() + K * 2.0 ** -24 * (a.abs() @ b.abs().T)
    for got in (lin(x), D.add_shares(lin.parts(x))):
        assert ((got.double() - a @ b.T).abs() <= bound).all()


@pytest.mark.parametrize("S", [2, 7, 16])
@pytest.mark.parametrize("W", [8, 1032, 4096, 8200])
def test_shares_meet_their_reader(S, W):
    """Shares of a product give what the stored product gives, bit for bit."""
    from quickstart_streaming_agents_amd.ops import ext
    g, T = gen(S + W), 5
    parts = rnd(g, S, T, W).to(DEV)
    y = D.add_shares(parts)
    w, post, table = (rnd(g, n, W, dtype=BF).to(DEV) for n in (1, 1, 9))
    ids = torch.tensor([0, 8, 3, 3, 1], device=DEV)
    res = rnd(g, T, W).to(DEV)
    for kw in ({}, {"post": post[0]}, {"layer": False, "post": post[0]},
               {"layer": False, "table": table, "ids": ids}, {"init": True}):
        for weight in (w[0], None):
            a, b = res.clone(), res.clone()
            got = D.residual_norm(a, parts, weight, None, 1e-5, **kw)
            want = D.residual_norm(b, y, weight, None, 1e-5, **kw)
            assert torch.equal(a, b) and torch.equal(got, want)
    for act in ("silu", "gelu"):
        assert torch.equal(D.glu_table(parts, table, ids, 0, act),
                           D.glu_table(y, table, ids, 0, act))
    a, b = (res.to(BF) for _ in range(2))
    got = D.rmsnorm_residual(parts, a, w[0], 1e-5)
    want = ext().rmsnorm_residual(y, b, w[0], 1e-5)
    assert torch.equal(a, b)
    # sums of squares in another order: one place of bf16
    close(got, want.cpu(), BF)
    odd = torch.empty(W + 1, dtype=BF, device=DEV)[1:].copy_(w[0])
    a, b = res.clone(), res.clone()
    assert torch.equal(D.residual_norm(a, parts, odd, None, 1e-5),
                       D.residual_norm(b, y, odd, None, 1e-5))


@pytest.mark.parametrize("dtype", [F32, BF])
@pytest.mark.parametrize("W", [4, 260, 4096])
def test_residual_norm_few_rows_or_many(W, dtype):
    """256 rows go as one round of loads each, 257 with a loop: alike, with
    whatever is given or absent, and what init replaces is not looked at."""
    g, T, V = gen(W), 257, 9
    res, y = rnd(g, T, W).to(DEV), rnd(g, T, W, dtype=dtype).to(DEV)
    w, b, vec, post, table = (rnd(g, n, W, dtype=dtype).to(DEV)
                              for n in (1, 1, 1, 1, V))
    ids = torch.arange(T, device=DEV) % V
    w, b, vec, post = w[0], b[0], vec[0], post[0]
    for branch, kw in ((y, {}), (y, {"post": post}), (None, {"vec": vec}),
                       (y, {"init": True}), (y, {"init": True, "post": post}),
                       (y, {"table": table, "tscale": .5}),
                       (y, {"table": table, "vec": vec, "post": post}),
                       (None, {"init": True, "table": table})):
        for layer, weight, bias in ((True, w, b), (True, w, None),
                                    (False, w, None), (False, None, None)):
            if branch is None and weight is None:
                continue                            # refused
            many, few = res.clone(), res[:256].clone()
            if kw.get("init"):
                many.fill_(float("nan")), few.fill_(float("nan"))
            def go(r):
                n = len(r)
                k = {**kw, "ids": ids[:n]} if "table" in kw else kw
                return D.residual_norm(
                    r, None if branch is None else branch[:n], weight, bias,
                    1e-4, layer=layer, **k)
            want, got = go(many), go(few)
            close(few, many[:256].cpu(), F32)
            close(got, want[:256].cpu(), dtype)


@pytest.mark.parametrize("dtype", [F32, BF])
@pytest.mark.parametrize("W", [4, 260, 1024])
def test_residual_norm_bits_of_few_or_many(W, dtype):
    """Widths that one group a thread covers either way: not a bit of a row depends
    on how many there are."""
    g, T = gen(W), 257
    res, y = rnd(g, T, W).to(DEV), rnd(g, T, W, dtype=dtype).to(DEV)
    w, b, vec, post = (rnd(g, W, dtype=dtype).to(DEV) for _ in range(4))
    table, ids = rnd(g, 9, W, dtype=dtype).to(DEV), torch.arange(T, device=DEV) % 9
    for kw in ({}, {"vec": vec}, {"post": post}, {"post": post, "init": True},
               {"post": post, "vec": vec, "table": table, "tscale": .5}):
        for layer, weight, bias in ((True, w, b), (True, w, None),
                                    (False, w, b), (False, w, None),
                                    (False, None, None)):
            out = []
            for n in (T, T - 1):
                r = res[:n].clone()
                k = {**kw, "ids": ids[:n]} if "table" in kw else kw
                out.append((r, D.residual_norm(r, y[:n], weight, bias, 1e-4,
                                               layer=layer, **k)))
            (many, a), (few, c) = out
            assert torch.equal(many[:-1], few) and torch.equal(a[:-1], c)


def test_product_in_shares():
    """What is left in shares adds up to the product."""
    g = gen(3)
    x, w = rnd(g, 100, 8192, dtype=BF).to(DEV), rnd(g, 512, 8192, dtype=BF)
    w = w.to(DEV)
    parts = D.linear_parts(x, w)
    assert parts.dim() == 3 and parts.shape[0] > 1
    a, b = x.double(), w.double()
    bound = 2.0 ** -8 * (a @ b.T).abs() + \
        8192 * 2.0 ** -24 * (a.abs() @ b.abs().T)
    assert ((D.add_shares(parts).double() - a @ b.T).abs() <= bound).all()


def test_linear_of_rows_far_apart():
    """The kernel's offsets of a row have 32 bits; rows too far apart for them
    are the library's."""
    from quickstart_streaming_agents_amd.models.layers import Linear
    K, far = 16_384, 1 << 24
    w = rnd(gen(1), 1024, K, dtype=BF).to(DEV)
    store = torch.empty(32 * far + K, dtype=BF, device=DEV)
    for step in (far - 8, far):
        x = store.as_strided((33, K), (step, 1))
        x.copy_(rnd(gen(2), 33, K, dtype=BF))
        assert D.rows_linear_ok(x, w) == (step < far)
        a, b = x.double(), w.double()
        close(Linear(w)(x), (a @ b.T).cpu(), BF)


def test_linear_under_observation():
    """Derivatives, transforms, tracing, modes and autocast meet the library's
    product, which knows them all."""
    import torch.autograd.forward_ad as fwd
    from torch.fx.experimental.proxy_tensor import make_fx
    from quickstart_streaming_agents_amd.models.layers import Linear
    M, N, K = 40, 1024, 16_384
    x, t = (rnd(gen(s), M, K, dtype=BF).to(DEV) for s in (1, 2))
    w = rnd(gen(3), N, K, dtype=BF, scale=K ** -0.5).to(DEV)
    lin = Linear(w)
    plain, slope = (torch.nn.functional.linear(y, w) for y in (x, t))
    assert D.rows_linear_ok(x, w)

    with fwd.dual_level():
        out = fwd.unpack_dual(lin(fwd.make_dual(x, t)))
    assert torch.equal(out.primal, plain) and torch.equal(out.tangent, slope)
    out = torch.func.jvp(lin, (x,), (t,))
    assert torch.equal(out[0], plain) and torch.equal(out[1], slope)
    y = x.clone().requires_grad_()
    lin(y).backward(plain)
    close(y.grad, (plain.double() @ w.double()).cpu(), BF)

    seen = []
    torch.func.vmap(lambda y: seen.append(D.rows_linear_ok(y, w)) or y)(
        x.view(1, M, K))
    assert seen == [False]
    for f in (make_fx(lin)(x), torch.jit.trace(lambda y: lin(y), x)):
        assert torch.equal(f(t), slope)
    with torch.autocast("cuda", torch.float16):
        assert lin(x).dtype == torch.float16
    assert D.rows_linear_ok(x, w)
