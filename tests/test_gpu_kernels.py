"""Numerics: each HIP kernel vs its plain-PyTorch fp32 reference.

All tests are @pytest.mark.gpu (MI355X only).  Tolerances account for
bf16 I/O (rel ~1e-2 on normalized magnitudes).
"""

import numpy as np
import pytest
import torch

from quickstart_streaming_agents_amd.ops import cpu_ref

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ext():
    from quickstart_streaming_agents_amd.ops import ext as get_ext
    return get_ext()


def dev():
    return "cuda:0"


def test_rmsnorm(ext):
    torch.manual_seed(0)
    x = torch.randn(33, 4096, dtype=torch.bfloat16, device=dev())
    w = torch.randn(4096, dtype=torch.bfloat16, device=dev())
    y = ext.rmsnorm(x, w, 1e-5)
    ref = cpu_ref.rmsnorm_ref(x.cpu(), w.cpu())
    torch.testing.assert_close(y.float().cpu(), ref, atol=5e-2, rtol=5e-2)


@pytest.mark.parametrize("rows", [1, 4, 7])
@pytest.mark.parametrize("H", [8, 384, 512, 520, 1024, 1032])
def test_rmsnorm_narrow(ext, rows, H):
    """Rows of one wave, up to one and two groups and just beyond; a rounding
    to bf16 of the result and of the residual each."""
    g = torch.Generator().manual_seed(H + rows)
    x, res, w = (torch.randn(*s, generator=g).bfloat16()
                 for s in ((rows, H), (rows, H), (H,)))

    def norm(t):
        t = t.double()
        return t * (t.square().mean(-1, keepdim=True) + 1e-5).rsqrt() * \
            w.double()

    y = ext.rmsnorm(x.to(dev()), w.to(dev()), 1e-5).cpu().double()
    assert ((y - norm(x)).abs() <= 2 ** -8 * norm(x).abs() + 1e-6).all()
    r = res.to(dev())
    y = ext.rmsnorm_residual(x.to(dev()), r, w.to(dev()), 1e-5).cpu().double()
    total = (x.float() + res.float()).bfloat16()
    assert torch.equal(r.cpu(), total)
    want = norm(total)
    # the mean square is the exact sums': 2**-9 of rounding either way
    assert ((y - want).abs() <= 2 ** -7 * want.abs() + 1e-6).all()


def test_rmsnorm_residual(ext):
    torch.manual_seed(1)
    x = torch.randn(17, 4096, dtype=torch.bfloat16, device=dev())
    res = torch.randn(17, 4096, dtype=torch.bfloat16, device=dev())
    w = torch.randn(4096, dtype=torch.bfloat16, device=dev())
    ref_y, ref_res = cpu_ref.rmsnorm_ref(x.cpu(), w.cpu(), residual=res.cpu())
    y = ext.rmsnorm_residual(x, res, w, 1e-5)
    torch.testing.assert_close(y.float().cpu(), ref_y, atol=5e-2, rtol=5e-2)
    torch.testing.assert_close(res.float().cpu(), ref_res, atol=3e-2, rtol=3e-2)


def test_swiglu(ext):
    torch.manual_seed(2)
    g = torch.randn(64, 14336, dtype=torch.bfloat16, device=dev())
    u = torch.randn(64, 14336, dtype=torch.bfloat16, device=dev())
    y = ext.swiglu(g, u)
    ref = cpu_ref.swiglu_ref(g.cpu(), u.cpu())
    torch.testing.assert_close(y.float().cpu(), ref, atol=5e-2, rtol=5e-2)


def test_rope(ext):
    torch.manual_seed(3)
    B, QH, KVH, D = 9, 8, 2, 128
    cos_t, sin_t = cpu_ref.rope_tables(512, D)
    q = torch.randn(B, QH, D, dtype=torch.bfloat16, device=dev())
    k = torch.randn(B, KVH, D, dtype=torch.bfloat16, device=dev())
    pos = torch.randint(0, 512, (B,), dtype=torch.int32, device=dev())
    q_ref = cpu_ref.rope_ref(q.cpu(), pos.cpu(), cos_t, sin_t)
    k_ref = cpu_ref.rope_ref(k.cpu(), pos.cpu(), cos_t, sin_t)
    ext.rope_inplace(q, k, cos_t.to(dev()), sin_t.to(dev()), pos)
    torch.testing.assert_close(q.float().cpu(), q_ref, atol=3e-2, rtol=3e-2)
    torch.testing.assert_close(k.float().cpu(), k_ref, atol=3e-2, rtol=3e-2)


def test_softmax_rows(ext):
    torch.manual_seed(4)
    s = torch.randn(32, 1000, dtype=torch.float32, device=dev()) * 4
    ref = cpu_ref.softmax_rows_ref(s.cpu(), col_offset=500, causal=True)
    ext.softmax_rows_(s, 500, True)
    torch.testing.assert_close(s.cpu(), ref, atol=1e-5, rtol=1e-4)


def _make_paged_kv(B, KVH, D, seq_lens, npages_total):
    torch.manual_seed(7)
    kc = torch.randn(npages_total, KVH, D // 8, 64, 8, dtype=torch.bfloat16,
                     device=dev())
    vc = torch.randn(npages_total, KVH, D, 64, dtype=torch.bfloat16, device=dev())
    max_pages = max((s + 63) // 64 for s in seq_lens)
    bt = torch.zeros(B, max_pages, dtype=torch.int32, device=dev())
    nxt = 0
    for b, s in enumerate(seq_lens):
        for p in range((s + 63) // 64):
            bt[b, p] = nxt % npages_total
            nxt += 1
    return kc, vc, bt


def test_paged_attn_decode(ext):
    B, QH, KVH, D = 4, 32, 8, 128
    seq_lens = [1, 64, 129, 500]
    kc, vc, bt = _make_paged_kv(B, KVH, D, seq_lens, 64)
    q = torch.randn(B, QH, D, dtype=torch.bfloat16, device=dev())
    sl = torch.tensor(seq_lens, dtype=torch.int32, device=dev())
    scale = 1.0 / (D ** 0.5)
    out = ext.paged_attn_decode(q, kc, vc, bt, sl, scale)
    ref = cpu_ref.paged_attn_ref(q.cpu(), kc.cpu(), vc.cpu(), bt.cpu(),
                                 sl.cpu(), scale)
    torch.testing.assert_close(out.float().cpu(), ref, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("B,KVH,D,pages", [
    (20, 4, 128, 17),                        # two shares of a row
    (2, 2, 64, 17), (2, 2, 128, 32),         # three, four: the first round
    (2, 2, 128, 33), (1, 2, 64, 81)])        # five, eleven: and a loop
def test_paged_attn_shares_merged(ext, B, KVH, D, pages):
    """Shares of long rows, and short rows that leave most of theirs empty."""
    QH = 4 * KVH
    seq_lens = [pages * 64 - 5] + [1, 300][:B - 1] + [700] * (B - 3)
    kc, vc, bt = _make_paged_kv(B, KVH, D, seq_lens, 2 * pages)
    q = torch.randn(B, QH, D, dtype=torch.bfloat16, device=dev())
    sl = torch.tensor(seq_lens, dtype=torch.int32, device=dev())
    out = ext.paged_attn_decode(q, kc, vc, bt, sl, D ** -0.5)
    ref = cpu_ref.paged_attn_ref(q.cpu(), kc.cpu(), vc.cpu(), bt.cpu(),
                                 sl.cpu(), D ** -0.5)
    torch.testing.assert_close(out.float().cpu(), ref, atol=2e-2, rtol=2e-2)


def test_kv_append_then_attend(ext):
    B, QH, KVH, D = 2, 8, 2, 128
    seq_lens = [65, 120]
    kc, vc, bt = _make_paged_kv(B, KVH, D, seq_lens, 16)
    knew = torch.randn(B, KVH, D, dtype=torch.bfloat16, device=dev())
    vnew = torch.randn(B, KVH, D, dtype=torch.bfloat16, device=dev())
    sl = torch.tensor(seq_lens, dtype=torch.int32, device=dev())
    ext.kv_append(knew, vnew, kc, vc, bt, sl)
    # verify the append landed where the reference expects
    for b, s in enumerate(seq_lens):
        pos = s - 1
        page = int(bt[b, pos // 64])
        pin = pos % 64
        got_v = vc[page, :, :, pin].float().cpu()
        torch.testing.assert_close(got_v, vnew[b].float().cpu(), atol=1e-3,
                                   rtol=1e-3)
        got_k = kc[page, :, :, pin, :].reshape(KVH, D).float().cpu()
        torch.testing.assert_close(got_k, knew[b].float().cpu(), atol=1e-3,
                                   rtol=1e-3)


def test_kv_scatter(ext):
    KVH, D = 2, 128
    T = 100
    kc = torch.zeros(4, KVH, D // 8, 64, 8, dtype=torch.bfloat16, device=dev())
    vc = torch.zeros(4, KVH, D, 64, dtype=torch.bfloat16, device=dev())
    knew = torch.randn(T, KVH, D, dtype=torch.bfloat16, device=dev())
    vnew = torch.randn(T, KVH, D, dtype=torch.bfloat16, device=dev())
    slots = torch.arange(T, dtype=torch.int32, device=dev()) + 28
    ext.kv_scatter(knew, vnew, kc, vc, slots)
    t = 40
    slot = int(slots[t])
    got = vc[slot // 64, :, :, slot % 64].float().cpu()
    torch.testing.assert_close(got, vnew[t].float().cpu(), atol=1e-3, rtol=1e-3)


def test_topk_cosine(ext):
    torch.manual_seed(5)
    Q, N, D, k = 7, 20000, 1536, 3
    docs = torch.randn(N, D, device=dev())
    docs = docs / docs.norm(dim=-1, keepdim=True)
    qs = torch.randn(Q, D, device=dev())
    qs = qs / qs.norm(dim=-1, keepdim=True)
    s, i = ext.topk_cosine(qs, docs, k)
    rs, ri = cpu_ref.topk_cosine_ref(qs.cpu(), docs.cpu(), k)
    torch.testing.assert_close(s.cpu(), rs, atol=1e-4, rtol=1e-4)
    assert torch.equal(i.cpu(), ri)


@pytest.mark.parametrize("Q,N,D,k", [
    (1, 1, 4, 1), (3, 2, 30, 5), (1, 15, 33, 16), (16, 17, 64, 3),
    (17, 65, 36, 4), (2, 1000, 1536, 10), (5, 32_767, 40, 16),
    (9, 32_768, 28, 3), (16, 32_801, 31, 1), (33, 70_001, 32, 2)])
def test_topk_cosine_edges(ext, Q, N, D, k):
    """Small whole numbers: every score is exact, so scores, documents and the
    order of equal scores (ascending document) are pinned without tolerance.
    Scores of -2 and less are never reported."""
    g = torch.Generator().manual_seed(Q * 1000 + N + D)
    docs = torch.randint(-2, 3, (N, D), generator=g).float()
    qs = torch.randint(-2, 3, (Q, D), generator=g).float()
    if N > 3:
        docs[2] = float("nan")
        docs[3] = torch.where(qs[0] >= 0, 1.0, -1.0) * float("inf")
    s, i = ext.topk_cosine(qs.to(dev()), docs.to(dev()), k)
    full = (qs.double() @ docs.double().T).nan_to_num(
        -9e9, float("inf"), -9e9)        # an infinite score comes first
    order = torch.sort(full, dim=1, descending=True, stable=True)[1][:, :k]
    want_s = torch.full((Q, k), -2.0)
    want_i = torch.full((Q, k), -1, dtype=torch.int32)
    top = full.gather(1, order)
    ok = top > -2
    m = order.shape[1]
    want_s[:, :m][ok] = top[ok].float()
    want_i[:, :m][ok] = order[ok].int()
    assert torch.equal(s.cpu(), want_s)
    assert torch.equal(i.cpu(), want_i)


@pytest.mark.parametrize("Q,N,D,k", [
    (16, 32_767, 96, 3), (16, 32_768, 100, 3), (1, 32_785, 132, 16),  # 16 | 64
    (17, 8191, 160, 5), (17, 8192, 4, 5), (32, 8209, 124, 3),  # 16 | 48 x 32
    (33, 4095, 64, 3), (33, 4097, 28, 3), (48, 4128, 260, 16),  # 16 | 32 x 48
    (49, 4096, 128, 3), (64, 4143, 36, 2),
    (17, 196_608, 4, 5), (33, 131_104, 4, 5),     # 4096 lists, and one more
    (33, 5000, 27, 3), (17, 9000, 31, 3), (16, 33_000, 1, 3)])  # odd rows
def test_topk_cosine_blocks(ext, Q, N, D, k):
    """Either side of each choice of a block; rows that end at, before and behind
    a step of 32 numbers.  Small whole numbers: scores are exact.  Memory that
    the search takes is poisoned first: nothing of it may be left."""
    g = torch.Generator().manual_seed(Q * 1000 + N + D)
    docs = torch.randint(-2, 3, (N, D), generator=g).float()
    qs = torch.randint(-2, 3, (Q, D), generator=g).float()
    docs[2] = float("nan")
    docs[N - 1] = qs[Q - 1] * 3
    a, b = qs.to(dev()), docs.to(dev())
    stale = [torch.full((n,), float("nan"), device=dev())
             for n in (Q * N // 8, Q * N // 4, 1 << 12)]
    del stale
    s, i = ext.topk_cosine(a, b, k)
    full = (qs @ docs.T).nan_to_num(-9e9)
    full[full <= -2] = -float("inf")
    top, order = torch.sort(full, dim=1, descending=True, stable=True)
    some = top[:, :k] > -2
    assert torch.equal(s.cpu(), top[:, :k].where(some, torch.tensor(-2.0)))
    assert torch.equal(i.cpu(), order[:, :k].int().where(
        some, torch.tensor(-1, dtype=torch.int32)))
    both = ext.topk_cosine_packed(a, b, k)
    assert both.shape == (2, Q, k)
    assert torch.equal(both[0].view(torch.float32), s)
    assert torch.equal(both[1], i)


@pytest.mark.parametrize("N,Q,D,k", [
    (1, 1, 1536, 1), (5, 3, 7, 5), (64, 1, 1536, 3), (65, 17, 129, 16),
    (3000, 2, 1534, 3), (40_000, 8, 64, 4), (0, 2, 8, 1), (9, 0, 8, 2)])
def test_topk_of_host_queries(ext, N, Q, D, k):
    """Queries in numpy of any order and length, among them zero, one whose
    norm floats do not hold and, where it does not fit, a NaN or infinity."""
    g = torch.Generator().manual_seed(N + Q)
    docs = torch.nn.functional.normalize(
        torch.randn(N, D, generator=g), dim=1).to(dev())
    q = torch.randn(Q, D, generator=g).numpy() * 3
    if Q > 1:
        q[1] = 0
    if Q > 2:
        q[2] = 3e38
    with np.errstate(over="ignore"):
        norm = np.linalg.norm(q, axis=1, keepdims=True)
    unit = (q / np.maximum(norm, 1e-12)).astype(np.float32)
    want = ext.topk_cosine_packed(torch.from_numpy(unit).to(dev()), docs,
                                  k).cpu().numpy()
    for x in (q, np.asfortranarray(q), np.repeat(q, 2, 0)[::2], q.tolist()
              if Q else q):
        got = ext.topk_cosine_host(x, docs, k)
        assert got.shape == (2, Q, k)
        # the norm's last bit, which numpy rounds on the way
        np.testing.assert_allclose(got[0].view(np.float32),
                                   want[0].view(np.float32), rtol=0,
                                   atol=4e-7)
        if N <= 64:
            assert (got[1] == want[1]).all()
    for bad in (np.nan, np.inf, -np.inf):
        if Q:
            x = q.copy()
            x[-1, D // 2] = bad
            assert ext.topk_cosine_host(x, docs, k) is None
    with pytest.raises(RuntimeError):
        ext.topk_cosine_host(np.zeros((1, D + 1)), docs, k)
    with pytest.raises(RuntimeError):
        ext.topk_cosine_host(q, docs, 17)


def test_window_agg(ext):
    torch.manual_seed(6)
    n, nkeys, nwin = 50000, 7, 288
    win = 300_000
    ts = torch.randint(0, nwin * win, (n,), dtype=torch.int64, device=dev())
    key = torch.randint(0, nkeys, (n,), dtype=torch.int32, device=dev())
    val = torch.rand(n, dtype=torch.float32, device=dev()) * 100
    counts, sums = ext.window_agg(ts, key, val, 0, win, nwin, nkeys)
    rc, rs = cpu_ref.window_agg_ref(ts.cpu(), key.cpu(), val.cpu(), 0, win,
                                    nwin, nkeys)
    assert torch.equal(counts.cpu(), rc)
    torch.testing.assert_close(sums.cpu(), rs, atol=1e-1, rtol=1e-4)


@pytest.mark.parametrize("Q,N,k", [
    (3, 262_144, 16), (3, 262_145, 16),      # 4096 and 4097 lists of 64
    (17, 131_072, 5), (17, 131_073, 5),      # and of 32
    (1, 900_001, 16)])
def test_topk_cosine_many_lists(ext, Q, N, k):
    """More lists than one merge holds; the best documents all in the last
    list, in the first, in any.  Small whole numbers: exact."""
    g = torch.Generator().manual_seed(N)
    docs = torch.randint(-2, 3, (N, 4), generator=g).float()
    qs = torch.randint(1, 3, (Q, 4), generator=g).float()
    docs[-k:] = 3 + torch.arange(k).float()[:, None]
    if Q > 1:
        qs[1] = -qs[1]
        docs[:k] = -4.0
    s, i = ext.topk_cosine(qs.to(dev()), docs.to(dev()), k)
    full = qs @ docs.T
    full[full <= -2] = -float("inf")
    top, order = torch.sort(full, dim=1, descending=True, stable=True)
    assert torch.equal(s.cpu(), top[:, :k])
    assert torch.equal(i.cpu(), order[:, :k].int())


def _agg_values(kind, n, g):
    v = torch.rand(n, generator=g) * 90 + 5
    if kind == "signed":
        v = torch.randn(n, generator=g) * 50
        v[::7], v[1::7] = 0.0, -0.0
    elif kind == "edge":                  # 38 bits from the lowest to the highest
        v = torch.full((n,), 1.0 - 2.0 ** -24)
        v[1::2] = -(2.0 ** -38)
    elif kind == "beyond":                # 39
        v = torch.full((n,), 2.0 - 2.0 ** -23)
        v[1::2] = -(2.0 ** -38)
    elif kind == "denormal":
        v = torch.randint(-99, 99, (n,), generator=g).float() * 2.0 ** -149
    elif kind == "huge":
        v = v * 2.0 ** 100
    elif kind == "zero":
        v = v * 0
    return v


@pytest.mark.parametrize("n,nkeys,nwin", [
    (69_633, 20, 300),                   # the last chunk is one event
    (400_000, 300, 150), (262_145, 1000, 30)])
@pytest.mark.parametrize("kind", ["plain", "signed", "edge", "beyond",
                                  "denormal", "huge", "zero", "none"])
def test_window_agg_values(ext, n, nkeys, nwin, kind):
    """Chunks whose values are whole numbers of a common unit are summed as such,
    the others as floats.  A chunk's sum is rounded once, the chunks of a cell
    (some share of n / 4096 / nwin, and two more) are added in f32; float sums
    round for every event."""
    g = torch.Generator().manual_seed(n)
    win = 60_000
    ts = (torch.arange(n) * (nwin * win / n)).long()
    key = (torch.rand(n, generator=g) ** 2 * nkeys).int().clamp(max=nkeys - 1)
    key[5::1000], key[6::1000] = -1, nkeys        # of no key: not counted
    val = _agg_values(kind, n, g)
    ok = (key >= 0) & (key < nkeys)
    bad = val.clone()
    if kind == "plain":                  # nor do their values matter
        bad[~ok] = float("nan")
    c, s = ext.window_agg(ts.to(dev()), key.to(dev()),
                          None if kind == "none" else bad.to(dev()), 0, win,
                          nwin, nkeys)
    slot = (key.long() * nwin + ts // win)[ok]
    want = torch.zeros(nkeys * nwin, dtype=torch.int32).scatter_add_(
        0, slot, torch.ones_like(slot, dtype=torch.int32))
    assert torch.equal(c.cpu().view(-1), want)
    if kind == "none":
        assert not s.any()
        return
    total, size = (torch.zeros(nkeys * nwin, dtype=torch.float64).scatter_add_(
        0, slot, x[ok].double()) for x in (val, val.abs()))
    roundings = n / 4096 / nwin + 3
    if kind == "beyond":
        roundings = want
    err = (s.cpu().view(-1).double() - total).abs()
    assert (err <= size * roundings * 2.0 ** -24).all()


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_window_agg_not_finite(ext, bad):
    n, nkeys, nwin, win = 80_000, 20, 300, 1000
    ts = (torch.arange(n) * (nwin * win / n)).long()
    key = (torch.arange(n) % nkeys).int()
    val = torch.ones(n)
    val[40_003] = bad
    c, s = ext.window_agg(ts.to(dev()), key.to(dev()), val.to(dev()), 0, win,
                          nwin, nkeys)
    s = s.cpu()
    k, w = int(key[40_003]), int(ts[40_003]) // win
    assert not torch.isfinite(s[k, w])
    s[k, w] = c.cpu()[k, w]
    assert torch.equal(s, c.cpu().float())


@pytest.mark.parametrize("n,nkeys,nwin,shuffle", [
    (1, 1, 1, False), (255, 3, 2, True), (257, 6144, 1, False),
    (5000, 6145, 2, False),              # one key more than a block's cells
    (140_000, 40, 300, False), (140_000, 40, 300, True),
    (300_001, 1000, 7, False)])
def test_window_agg_edges(ext, n, nkeys, nwin, shuffle):
    """Chunks counted in LDS and chunks that go to memory directly; events
    before and behind the windows.  Whole values: sums are exact."""
    g = torch.Generator().manual_seed(n)
    win, t0 = 1000 + n % 7, 5000 - (n % 3) * (1 << 40)
    ts = torch.randint(t0 - 2 * win, t0 + (nwin + 1) * win, (n,), generator=g)
    if not shuffle:
        ts = ts.sort()[0]
    key = torch.randint(0, nkeys, (n,), generator=g, dtype=torch.int32)
    val = torch.randint(-8, 9, (n,), generator=g).float()
    w = torch.div(ts - t0, win, rounding_mode="trunc")
    ok = (w >= 0) & (w < nwin)
    at = (key.long() * nwin + w)[ok]
    counts = torch.zeros(nkeys * nwin, dtype=torch.int32).index_add_(
        0, at, torch.ones_like(at, dtype=torch.int32)).view(nkeys, nwin)
    sums = torch.zeros(nkeys * nwin).index_add_(0, at, val[ok]) \
        .view(nkeys, nwin)
    args = (t0, win, nwin, nkeys)
    c, s = ext.window_agg(ts.to(dev()), key.to(dev()), val.to(dev()), *args)
    assert torch.equal(c.cpu(), counts) and torch.equal(s.cpu(), sums)
    c, s = ext.window_agg(ts.to(dev()), key.to(dev()), None, *args)
    assert torch.equal(c.cpu(), counts) and not s.any()


@pytest.mark.parametrize("nkeys,nwin", [(1, 1), (511, 1), (1, 513),
                                        ((1 << 21) + 1, 16),
                                        ((1 << 21) + 1, 17)])
def test_window_agg_clears_its_tables(ext, nkeys, nwin):
    """Around the 1024 cells of a block and the 67,108,864 of a full grid: nothing of
    what the memory held before is left, to the last cell."""
    dirty = torch.ones(2, nkeys, nwin, dtype=torch.int32, device=dev())
    del dirty                                   # its block is the next one given
    ts = torch.tensor([0, 10 * nwin - 1], device=dev())
    key = torch.tensor([0, nkeys - 1], dtype=torch.int32, device=dev())
    val = torch.tensor([2., 3.], device=dev())
    counts, sums = ext.window_agg(ts, key, val, 0, 10, nwin, nkeys)
    assert int(counts.sum()) == 2 and float(sums.double().sum()) == 5
    assert int(torch.count_nonzero(counts)) <= 2
    assert int(torch.count_nonzero(sums)) <= 2
    assert int(counts[-1, -1]) >= 1 and float(sums[-1, -1]) >= 3


@pytest.mark.parametrize("n,nkeys,nwin", [
    (131_072, 40, 200), (131_073, 40, 200),    # chunks of 256, of 1024
    (140_000, 2049, 3), (262_144, 40, 154),
    (262_145, 40, 154),                        # merged, 65 chunks
    (65_536, 2048, 3), (65_537, 2048, 3),      # the whole table fits
    (300_000, 6144, 44), (300_000, 6144, 43),  # six in ten chunks fit
    (300_000, 6145, 1), (270_000, 4_200_000, 2),
    (8_400_000, 10, 50)])                      # longer chunks
def test_window_agg_forms(ext, n, nkeys, nwin):
    """Both sides of the rule that chooses a form, events in order and not, and
    more keys than a launch of the merge has rows for.  Whole values."""
    g = torch.Generator().manual_seed(n + nkeys)
    ts = torch.randint(-500, nwin * 1000 + 500, (n,), generator=g)
    key = torch.randint(-1, nkeys + 1, (n,), generator=g, dtype=torch.int32)
    key[:2] = torch.tensor([0, nkeys - 1])
    val = torch.randint(-8, 9, (n,), generator=g).float()
    for order in (ts.sort()[0], ts):
        w = torch.div(order, 1000, rounding_mode="trunc")
        ok = (w < nwin) & (key >= 0) & (key < nkeys)
        at = (key.long() * nwin + w)[ok]
        counts = torch.zeros(nkeys * nwin, dtype=torch.int32).index_add_(
            0, at, torch.ones_like(at, dtype=torch.int32))
        sums = torch.zeros(nkeys * nwin).index_add_(0, at, val[ok])
        c, s = ext.window_agg(order.to(dev()), key.to(dev()), val.to(dev()),
                              0, 1000, nwin, nkeys)
        assert torch.equal(c.cpu().view(-1), counts)
        assert torch.equal(s.cpu().view(-1), sums)


@pytest.mark.parametrize("n", [1, 5, 6, 9, 12, 20, 63, 64, 69, 288, 7000])
def test_anomaly_batch_lengths(ext, n):
    """Every order of the fit (0 to 4 lags) at lengths around the wave."""
    from quickstart_streaming_agents_amd.runtime.anomaly import ar_forecast
    rng = np.random.default_rng(n)
    x = rng.normal(100, 10, (5, n + 3)).astype(np.float32)
    x[:, n:] = 1e9                       # beyond the length: never read
    fc, se, dof = ext.anomaly_batch(
        torch.from_numpy(x).to(dev()),
        torch.full((5,), n, dtype=torch.int32, device=dev()), 4)
    for i in range(5):
        f, e, d = ar_forecast(x[i, :n].astype(np.float64), 4)
        # f32 sums over n values about 100: the centred products keep 5 digits
        assert abs(float(fc[i]) - f) < 1e-3 * abs(f)
        assert abs(float(se[i]) - e) < 2e-3 * e
        assert int(dof[i]) == d


def test_hash_table_as_two_arrays(ext):
    """A table's words may be kept as separate arrays."""
    keys = torch.arange(1000, dtype=torch.int64, device=dev()) * 7919
    ts = torch.arange(1000, dtype=torch.int64, device=dev()) - 5
    k, p = ext.hash_build(keys, ts)
    probe = torch.cat([keys.flip(0), keys + 1])
    for cut in (-1, 3, 1 << 50):
        rows = ext.hash_probe(k, p, probe, cut)
        assert torch.equal(rows, ext.hash_probe(k.clone(), p.clone(), probe,
                                                cut))
        want = torch.where(ts.clamp(min=0) >= cut,
                           torch.arange(1000, device=dev()), -1).flip(0)
        assert torch.equal(rows[:1000].long(), want)
        assert (rows[1000:] == -1).all()


# half full where n is a power of two; steps of one beyond 131072 rows
@pytest.mark.parametrize("n", [1, 32, 33, 1024, 131_072, 131_073])
def test_hash_table_fill(ext, n):
    g = torch.Generator(device=dev()).manual_seed(n)
    keys = torch.randperm(4 * n, generator=g, device=dev()) * 3 - n
    ts = torch.randint(0, 1000, (n,), generator=g, device=dev())
    k, p = ext.hash_build(keys[:n], ts)
    rows = ext.hash_probe(k, p, keys, 500)
    want = torch.where(ts >= 500, torch.arange(n, device=dev()), -1)
    assert torch.equal(rows[:n].long(), want)
    assert (rows[n:] == -1).all()


@pytest.mark.parametrize("n", [61, 62, 509, 510])     # rows of 64, 512 and more
def test_anomaly_batch_staged(ext, n):
    test_anomaly_batch_lengths(ext, n)


@pytest.mark.parametrize("T", [7, 128, 129])
def test_anomaly_batch_of_many_series(ext, T):
    """Series read from memory or from LDS, either side of that rule: the same
    sums in the same order."""
    g = torch.Generator().manual_seed(T)
    x = torch.rand(8193, T, generator=g).to(dev())
    n = torch.randint(0, T + 1, (8193,), generator=g).int().to(dev())
    n[:2] = T
    many = ext.anomaly_batch(x, n, 4)
    few = ext.anomaly_batch(x[:8192], n[:8192], 4)
    for a, b in zip(many, few):
        assert torch.equal(a[:8192], b)


def test_anomaly_batch_matches_cpu(ext):
    from quickstart_streaming_agents_amd.runtime.anomaly import ar_forecast
    rng = np.random.default_rng(0)
    K, Tmax = 16, 400
    series = np.zeros((K, Tmax), dtype=np.float32)
    lengths = np.zeros(K, dtype=np.int32)
    for kk in range(K):
        n = int(rng.integers(10, Tmax))
        lengths[kk] = n
        base = rng.uniform(10, 1000)
        series[kk, :n] = base + rng.normal(0, base * 0.02, n).astype(np.float32)
    s_t = torch.from_numpy(series).to(dev())
    l_t = torch.from_numpy(lengths).to(dev())
    fc, se, dof = ext.anomaly_batch(s_t, l_t, 4)
    for kk in range(K):
        f_ref, se_ref, dof_ref = ar_forecast(
            series[kk, :lengths[kk]].astype(np.float64), 4)
        assert dof[kk].item() == dof_ref
        assert abs(fc[kk].item() - f_ref) < max(3e-3 * abs(f_ref), 1e-2)
        assert abs(se[kk].item() - se_ref) < max(0.05 * se_ref, 1e-2)


def test_skinny_gemm_matches_linear():
    """Weight-streaming decode GEMM vs fp32 reference: both split-K (small
    N) and single-pass (large N) paths, ragged M."""
    import torch.nn.functional as F
    from quickstart_streaming_agents_amd.ops import ext
    torch.manual_seed(3)
    for M, N, K in [(24, 4096, 4096), (1, 512, 512), (32, 1024, 256),
                    (17, 28672, 512)]:
        a = torch.randn(M, K, device="cuda:0", dtype=torch.bfloat16) * 0.5
        w = torch.randn(N, K, device="cuda:0", dtype=torch.bfloat16) * 0.02
        wf = ext().pack_weight_frag(w)
        out = ext().skinny_gemm(a, wf, N, K)
        ref = a.float() @ w.float().T
        err = (out.float() - ref).abs().max().item()
        scale = ref.abs().max().item() + 1e-6
        assert err / scale < 2e-2, f"M{M} N{N} K{K}: rel err {err/scale}"


def test_skinny_gemm_strided_rows():
    """Row-strided activations (views into a larger buffer) work."""
    from quickstart_streaming_agents_amd.ops import ext
    torch.manual_seed(4)
    buf = torch.randn(8, 1024, device="cuda:0", dtype=torch.bfloat16)
    a = buf[:, :512]
    w = torch.randn(256, 512, device="cuda:0", dtype=torch.bfloat16) * 0.05
    wf = ext().pack_weight_frag(w)
    out = ext().skinny_gemm(a.contiguous(), wf, 256, 512)
    ref = a.float() @ w.float().T
    assert (out.float() - ref).abs().max().item() < 2e-2 * (
        ref.abs().max().item() + 1e-6)


def test_softmax_rows_bf16_matches_ref():
    from quickstart_streaming_agents_amd.ops import dispatch as D
    torch.manual_seed(9)
    rows, cols = 300, 256
    scores = torch.randn(rows, cols, device="cuda:0",
                         dtype=torch.bfloat16) * 4
    limits = torch.randint(0, cols + 1, (rows,), dtype=torch.int32,
                           device="cuda:0")
    ref = scores.clone().cpu()
    lim_cpu = limits.cpu()
    D.softmax_rows_bf16_(ref, 0.125, lim_cpu)          # CPU reference path
    D.softmax_rows_bf16_(scores, 0.125, limits)        # HIP kernel
    got = scores.cpu().float()
    torch.testing.assert_close(got, ref.float(), atol=2e-2, rtol=2e-2)
    # beyond-limit strictly zero; rows sum to ~1 where limit > 0
    for r in (0, 7, 123):
        lim = int(lim_cpu[r])
        assert (got[r, lim:] == 0).all()
        if lim > 0:
            assert abs(got[r, :lim].sum().item() - 1.0) < 2e-2


def test_rope_kv_append_matches_composed(ext):
    """Fused rope+append == rope_inplace followed by kv_append."""
    import copy
    torch.manual_seed(6)
    B, QH, KVH, D = 5, 8, 2, 128
    from quickstart_streaming_agents_amd.ops import cpu_ref
    cos_t, sin_t = cpu_ref.rope_tables(256, D)
    cos_t, sin_t = cos_t.to(dev()), sin_t.to(dev())
    seq_lens = torch.tensor([3, 64, 65, 1, 120], dtype=torch.int32,
                            device=dev())
    npages = 3
    bt = torch.arange(B * npages, dtype=torch.int32,
                      device=dev()).reshape(B, npages)
    q = torch.randn(B, QH, D, dtype=torch.bfloat16, device=dev())
    k = torch.randn(B, KVH, D, dtype=torch.bfloat16, device=dev())
    v = torch.randn(B, KVH, D, dtype=torch.bfloat16, device=dev())
    kc1 = torch.zeros(B * npages, KVH, D // 8, 64, 8, dtype=torch.bfloat16,
                      device=dev())
    vc1 = torch.zeros(B * npages, KVH, D, 64, dtype=torch.bfloat16,
                      device=dev())
    kc2, vc2 = kc1.clone(), vc1.clone()

    # composed reference
    q2, k2 = q.clone(), k.clone()
    pos = (seq_lens - 1).clamp(min=0).int()
    ext.rope_inplace(q2, k2, cos_t, sin_t, pos)
    ext.kv_append(k2, v, kc2, vc2, bt, seq_lens)
    # fused
    q1 = q.clone()
    ext.rope_kv_append(q1, k, v, kc1, vc1, cos_t, sin_t, bt, seq_lens)

    torch.testing.assert_close(q1, q2)
    torch.testing.assert_close(kc1, kc2)
    torch.testing.assert_close(vc1, vc2)


def test_paged_attention_forced_rescale(ext):
    """Force the online-softmax rescale with per-head divergent maxima at
    a LATE page (guide rule: a rare data-dependent branch needs its own
    test) — this catches per-row/column alpha mix-ups the random-data
    test cannot."""
    torch.manual_seed(8)
    B, QH, KVH, D = 2, 8, 2, 128
    seqlen = 3 * 64  # 3 pages
    kc = torch.randn(8, KVH, D // 8, 64, 8, dtype=torch.bfloat16,
                     device=dev()) * 0.3
    vc = torch.randn(8, KVH, D, 64, dtype=torch.bfloat16, device=dev())
    q = torch.randn(B, QH, D, dtype=torch.bfloat16, device=dev())
    # spike K at page 2 position 7 so scores jump there; make q for SOME
    # heads align with the spike direction and others anti-align
    spike = torch.randn(D, device=dev(), dtype=torch.bfloat16) * 3
    kc[2 + 3, :, :, 7, :] = spike.reshape(D // 8, 8).unsqueeze(0) * 2
    kc[2, :, :, 7, :] = spike.reshape(D // 8, 8).unsqueeze(0) * 2
    for h in range(QH):
        sgn = 1.0 if h % 2 == 0 else -1.0
        q[:, h] = sgn * spike + torch.randn(D, device=dev(),
                                            dtype=torch.bfloat16) * 0.2
    bt = torch.tensor([[0, 1, 2], [3, 4, 5]], dtype=torch.int32,
                      device=dev())
    sl = torch.tensor([seqlen, seqlen - 10], dtype=torch.int32,
                      device=dev())
    out = ext.paged_attn_decode(q, kc, vc, bt, sl, 0.088)
    ref = cpu_ref.paged_attn_ref(q.cpu(), kc.cpu(), vc.cpu(), bt.cpu(),
                                 sl.cpu(), 0.088)
    torch.testing.assert_close(out.float().cpu(), ref.float(), atol=4e-2,
                               rtol=4e-2)


def test_skinny_gemm_fp8_matches_dequant_ref():
    """fp8 (e4m3, per-channel W8A16) decode GEMM vs the dequantized fp32
    reference: the in-kernel cvt_pk_f32_fp8 + perm pack is exact, so the
    only tolerance is MFMA accumulation order."""
    from quickstart_streaming_agents_amd.ops import dispatch as D
    from quickstart_streaming_agents_amd.ops import ext
    torch.manual_seed(5)
    for M, N, K in [(24, 4096, 4096), (1, 512, 512), (32, 1024, 256),
                    (17, 28672, 512), (24, 128, 14336)]:
        a = torch.randn(M, K, device="cuda:0", dtype=torch.bfloat16) * 0.5
        w = torch.randn(N, K, device="cuda:0", dtype=torch.bfloat16) * 0.02
        qf, s = D.pack_weight_fp8(w)
        out = ext().skinny_gemm_fp8(a, qf, s, N, K)
        wd = D.unpack_weight_fp8(qf, s, N, K)      # exact dequant (f32)
        ref = a.float() @ wd.T
        err = (out.float() - ref).abs().max().item()
        scale = ref.abs().max().item() + 1e-6
        assert err / scale < 2e-2, f"M{M} N{N} K{K}: rel err {err/scale}"
        # quantization error vs the unquantized weights is bounded (e4m3
        # per-channel: ~0.5-3% on random normal weights)
        ref_bf = a.float() @ w.float().T
        qerr = (out.float() - ref_bf).abs().max().item() / \
            (ref_bf.abs().std().item() + 1e-6)
        assert qerr < 0.5, f"quantization error blew up: {qerr}"


def test_skinny_gemm_fp8_every_code():
    """Each of the 256 codes comes out as the bf16 value it stands for, the
    subnormal ones and NaN too."""
    from quickstart_streaming_agents_amd.ops import ext
    codes = torch.arange(256, dtype=torch.uint8)
    q = codes[:, None].expand(256, 256).contiguous()     # a row of W per code
    qf = q.reshape(16, 16, 4, 2, 4, 8).permute(0, 2, 1, 4, 3, 5).contiguous()
    a = torch.zeros(3, 256, dtype=torch.bfloat16)
    a[0, 0] = a[1, 77] = a[2, 255] = 1
    out = ext().skinny_gemm_fp8(a.cuda(), qf.cuda(), torch.ones(256).cuda(),
                                256, 256).cpu()
    want = codes.view(torch.float8_e4m3fn).float()
    assert torch.equal(out.float().nan_to_num(nan=1e3),
                       want.nan_to_num(nan=1e3).expand(3, 256))


@pytest.mark.parametrize("K", [256, 512, 768, 1024, 1280, 3328, 7168])
@pytest.mark.parametrize("M", [1, 3, 4, 5, 8, 9, 17])
def test_skinny_fp8_steps(M, K):
    """Numbers of steps that the groups of a block's waves do not divide: all forms
    against f64, rows of A in a wider matrix and off its 16 bytes."""
    from quickstart_streaming_agents_amd.ops import dispatch as D
    from quickstart_streaming_agents_amd.ops import ext
    g = torch.Generator(device="cuda").manual_seed(K + M)
    N, eps = 128, 1e-5
    w = torch.randn(N, K, generator=g, device="cuda").bfloat16() * 0.05
    packed = D.pack_weight_fp8(w)
    W = D.unpack_weight_fp8(*packed, N, K).double()
    wide = torch.full((M, K + 24), float("nan"), device="cuda").bfloat16()
    wide[:, 8:K + 8] = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    x = wide[:, 8:K + 8]
    want = x.double() @ W.t()

    def close(got, want):
        # sums of K products in f32, rounded to bf16: 2^-9 of a value
        err = (got.double() - want).norm()
        assert err <= 4e-3 * want.norm(), float(err / want.norm())

    close(ext().skinny_gemm_fp8(x, *packed, N, K), want)
    off = torch.full((M * K + 3,), float("nan"), device="cuda").bfloat16()
    off[3:] = x.reshape(-1)
    close(ext().skinny_gemm_fp8(off[3:].view(M, K), *packed, N, K), want)
    # steps of the decoder: rows with their norm, and with the residual
    embed = torch.randn(50, K, generator=g, device="cuda").bfloat16()
    ids = torch.randint(0, 50, (M,), generator=g, device="cuda")
    ones = torch.ones(K, device="cuda").bfloat16()
    res, rows, ss = D.embed_rows(embed, ids, ones)
    h = embed[ids].double()
    y = h * torch.rsqrt(h.square().mean(-1, keepdim=True) + eps) @ W.t()
    close(D.norm_linear_fp8(rows, ss, 1, M, eps, packed, N, K), y)
    old = torch.randn(M, N, generator=g, device="cuda").bfloat16()
    new = old.clone()
    D.linear_residual_fp8(rows, packed, N, K, new,
                          torch.ones(N, device="cuda").bfloat16())
    close(new, old.double() + h @ W.t())


def test_skinny_rows_and_weights_anywhere(ext):
    """Rows off the 16 bytes that a load takes, an odd number of elements or some
    2^31 bytes apart, and weights off their 16 bytes, give the bits of a copy."""
    from quickstart_streaming_agents_amd.ops import dispatch as D
    from quickstart_streaming_agents_amd.ops import lm_ext
    M, N, K = 3, 64, 512
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = torch.randn(N, K, generator=g, device="cuda").bfloat16()
    wf, (qf, scale) = ext.pack_weight_frag(w), D.pack_weight_fp8(w)

    def moved(t, by):
        flat = t.new_empty(t.numel() + by)[by:]
        return flat.copy_(t.reshape(-1)).view(t.shape)

    def strided(step):
        flat = x.new_empty((M - 1) * step + K)
        return flat.as_strided((M, K), (step, 1)).copy_(x)

    far = 1 << 29
    rows = [moved(x, 3), strided(K + 5), strided(far)]
    calls = [(ext.skinny_gemm, (wf,)), (ext.skinny_gemm_fp8, (qf, scale))]
    for call, (packed, *more) in calls:
        want = call(x, packed, *more, N, K)
        for a in rows:
            assert torch.equal(call(a, packed, *more, N, K), want)
        assert torch.equal(call(x, moved(packed, 1), *more, N, K), want)
    want = lm_ext().skinny_gemm(x, wf, N, K, False)
    for a, b in ((strided(far), wf), (x, moved(wf, 1))):
        assert torch.equal(lm_ext().skinny_gemm(a, b, N, K, False), want)
    # rows of a step
    embed, ids = x, torch.arange(M, device="cuda")
    ones = torch.ones(K, device="cuda").bfloat16()
    old = torch.randn(M, N, generator=g, device="cuda").bfloat16()
    _, step, ss = D.embed_rows(embed, ids, ones)

    def both(step, qf):
        res = old.clone()
        D.linear_residual_fp8(step, (qf, scale), N, K, res, ones[:N])
        return D.norm_linear_fp8(step, ss, 1, M, 1e-5, (qf, scale), N, K), res

    want = both(step, qf)
    for a, b in ((moved(step, 1), qf), (step, moved(qf, 1))):
        assert all(map(torch.equal, both(a, b), want))


@pytest.mark.parametrize("K", [256, 768, 1280, 4096, 7168])
@pytest.mark.parametrize("M", [2, 3, 4, 5, 17])
def test_skinny_fp8_rows_apart(M, K):
    """A row of NaN or of infinities, and such rows before and behind those given,
    change no bit of the others: what is read beyond the last step is zero for
    every row, in all forms."""
    from quickstart_streaming_agents_amd.ops import dispatch as D
    from quickstart_streaming_agents_amd.ops import ext
    g = torch.Generator(device="cuda").manual_seed(K + M)
    N = 128
    w = torch.randn(N, K, generator=g, device="cuda").bfloat16() * 0.05
    packed = D.pack_weight_fp8(w)
    ids = torch.arange(M, device="cuda")
    ones = torch.ones(max(N, K), device="cuda").bfloat16()
    rows = torch.randn(M + 2, K, generator=g, device="cuda").bfloat16()
    old = torch.randn(M, N, generator=g, device="cuda").bfloat16()

    def run(bad, value):
        t = rows.clone()
        t[0] = t[-1] = float("nan")
        if value is not None:
            t[1 + bad] = value
        x = t[1:-1]
        out = [ext().skinny_gemm_fp8(x, *packed, N, K)]
        _, step, ss = D.embed_rows(x.contiguous(), ids, ones[:K])
        out.append(D.norm_linear_fp8(step, ss, 1, M, 1e-5, packed, N, K))
        out.append(old.clone())
        D.linear_residual_fp8(step, packed, N, K, out[-1], ones[:N])
        return [torch.cat((o[:bad], o[bad + 1:])) for o in out]

    for bad in (0, M - 1):
        want = run(bad, None)
        assert all(torch.isfinite(t).all() for t in want)
        for value in (float("nan"), float("inf")):
            assert all(map(torch.equal, run(bad, value), want))


def test_skinny_gemm_fp8_gpu_pack_matches_cpu_pack():
    """CPU and GPU packs agree in VALUE (the f32->e4m3 cast may round
    ties differently across backends; one e4m3 quantum of slack)."""
    from quickstart_streaming_agents_amd.ops import dispatch as D
    torch.manual_seed(6)
    w = torch.randn(64, 512, dtype=torch.bfloat16) * 0.02
    qf_cpu, s_cpu = D.pack_weight_fp8(w)
    qf_gpu, s_gpu = D.pack_weight_fp8(w.cuda())
    assert torch.allclose(s_cpu, s_gpu.cpu())
    wd_cpu = D.unpack_weight_fp8(qf_cpu, s_cpu, 64, 512)
    wd_gpu = D.unpack_weight_fp8(qf_gpu.cpu(), s_gpu.cpu(), 64, 512)
    # quantum = scale * 2^-3 at the value's binade; bound by per-channel
    # scale * max step (values <= 448 * s -> step <= 32 * s)
    step = (s_cpu[:, None] * 32.0)
    assert ((wd_cpu - wd_gpu).abs() <= step + 1e-12).all()
    frac_diff = (qf_cpu != qf_gpu.cpu()).float().mean().item()
    assert frac_diff < 0.02, f"packs differ on {frac_diff:.1%} of bytes"


def _step_rows(x):
    """[M, K] in the layout that decoding steps pass between projections."""
    M, K = x.shape
    if M <= 4:
        return x.contiguous()
    mt = 1 if M <= 16 else 2
    p = torch.full((mt * 16, K), float("nan"), dtype=x.dtype, device=x.device)
    p[:M] = x
    return p.view(mt, 16, K // 32, 4, 8).permute(2, 0, 3, 1, 4) \
        .reshape(K // 32, mt, 64, 8).contiguous()


def _from_step_rows(x, M):
    if x.dim() == 2:
        return x
    kb, mt = x.shape[:2]
    return x.view(kb, mt, 4, 16, 8).permute(1, 3, 0, 2, 4) \
        .reshape(mt * 16, kb * 32)[:M]


@pytest.mark.parametrize("M", [1, 4, 5, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(64, 256), (192, 768), (4096, 8448),
                                 (65_600, 512), (6208, 2304)])
def test_skinny_fp8_forms(M, N, K):
    """Plain, normed, gated and residual forms against f64 on the
    dequantized weights; rows that do not exist hold NaN."""
    from quickstart_streaming_agents_amd.ops import dispatch as D
    from quickstart_streaming_agents_amd.ops import ext
    torch.manual_seed(M + N + K)
    w = torch.randn(N, K, device=dev(), dtype=torch.bfloat16) * K ** -0.5
    packed = D.pack_weight_fp8(w)
    W = D.unpack_weight_fp8(*packed, N, K).double()
    x = torch.randn(M, K + 64, device=dev(), dtype=torch.bfloat16)[:, :K]
    # operands are exact here; results are rounded to bf16 (2^-9 each)
    tol = 2 ** -8

    def close(got, want):
        err = (got.double() - want).norm() / want.norm()
        assert err < tol, float(err)

    y = x.double() @ W.T
    close(ext().skinny_gemm_fp8(x, *packed, N, K), y)
    xs = _step_rows(x)
    eps = 1e-5
    for parts in (1, 3, 260):
        p4 = (parts + 3) // 4 * 4
        ss = torch.full((32, p4), float("nan"), device=dev())
        share = torch.rand(M, parts, device=dev())
        ss[:M, :parts] = share / share.sum(1, keepdim=True) \
            * x.float().square().sum(1, keepdim=True)
        h = y * torch.rsqrt(x.double().square().mean(1, keepdim=True) + eps)
        close(D.norm_linear_fp8(xs, ss, parts, M, eps, packed, N, K), h)
        g, u = h.chunk(2, 1)
        act = D.norm_linear_fp8(xs, ss, parts, M, eps, packed, N, K, glu=True)
        close(_from_step_rows(act, M), torch.nn.functional.silu(g) * u)
    res = torch.randn(M, N, device=dev(), dtype=torch.bfloat16)
    nw = (1 + 0.2 * torch.randn(N, device=dev())).bfloat16()
    want = res.double() + y
    nxt, out = D.linear_residual_fp8(xs, packed, N, K, res, nw)
    close(res, want)
    assert torch.equal(_from_step_rows(nxt, M),
                       (res.float() * nw.float()).bfloat16())
    sums = out[:M, :N // 16].double().sum(1)
    assert ((sums - want.square().sum(1)).abs()
            < tol * want.square().sum(1)).all()


@pytest.mark.parametrize("M", [8, 9, 16, 17])
@pytest.mark.parametrize("N,K", [(12288, 1024), (12352, 2048), (16384, 2304),
                                 (28672, 2304), (28736, 2304)])
def test_skinny_fp8_wide_blocks(M, N, K):
    """Plain and gated forms about where a block takes four tiles of columns."""
    from quickstart_streaming_agents_amd.ops import dispatch as D
    torch.manual_seed(M + N + K)
    w = torch.randn(N, K, device=dev(), dtype=torch.bfloat16) * K ** -0.5
    packed = D.pack_weight_fp8(w)
    x = torch.randn(M, K, device=dev(), dtype=torch.bfloat16)
    ss = torch.full((32, 4), float("nan"), device=dev())
    ss[:M, 0] = x.float().square().sum(1)
    h = x.double() @ D.unpack_weight_fp8(*packed, N, K).double().T \
        * torch.rsqrt(x.double().square().mean(1, keepdim=True) + 1e-5)
    got = D.norm_linear_fp8(_step_rows(x), ss, 1, M, 1e-5, packed, N, K)
    assert (got.double() - h).norm() < 2 ** -8 * h.norm()   # rounded to bf16
    act = D.norm_linear_fp8(_step_rows(x), ss, 1, M, 1e-5, packed, N, K,
                            glu=True)
    g, u = h.chunk(2, 1)
    want = torch.nn.functional.silu(g) * u
    assert (_from_step_rows(act, M).double() - want).norm() \
        < 2 ** -8 * want.norm()


@pytest.mark.parametrize("M", [1, 3, 4, 5, 8, 9])
@pytest.mark.parametrize("N,K", [(32, 3072), (2048, 3328), (224, 5888),
                                 (992, 6144), (2048, 8192), (2080, 8192)])
def test_skinny_fp8_half_tiles(M, N, K):
    """The residual form of few columns in half tiles, and on either side of
    where they are taken; rows that do not exist hold NaN, and the norm that
    follows reads the parts."""
    from quickstart_streaming_agents_amd.ops import dispatch as D
    torch.manual_seed(M + N + K)
    w = torch.randn(N, K, device=dev(), dtype=torch.bfloat16) * K ** -0.5
    packed = D.pack_weight_fp8(w)
    W = D.unpack_weight_fp8(*packed, N, K).double()
    x = torch.randn(M, K, device=dev(), dtype=torch.bfloat16)
    res = torch.randn(M, N, device=dev(), dtype=torch.bfloat16)
    nw = (1 + 0.2 * torch.randn(N, device=dev())).bfloat16()
    want = res.double() + x.double() @ W.T
    nxt, ss = D.linear_residual_fp8(_step_rows(x), packed, N, K, res, nw)
    # operands are exact, sums f32 (K 2^-24), the result rounded (2^-9)
    assert ((res.double() - want).abs() <= 2 ** -8 * want.abs()
            + K * 2 ** -24 * (x.double().abs() @ W.abs().T)).all()
    assert torch.equal(_from_step_rows(nxt, M),
                       (res.float() * nw.float()).bfloat16())
    parts = D.residual_parts_fp8(M, N, K)
    assert parts == N // (8 if M <= 8 and N <= 2048 else 16)
    assert ss.shape == (32, -(-parts // 4) * 4)
    sums = ss[:M, :parts].double().sum(1)
    assert ((sums - want.square().sum(1)).abs()
            < 2 ** -8 * want.square().sum(1)).all()
    if N % 256 == 0:
        v = torch.randn(64, N, device=dev(), dtype=torch.bfloat16) * N ** -0.5
        p2 = D.pack_weight_fp8(v)
        got = D.norm_linear_fp8(nxt, ss, parts, M, 1e-5, p2, 64, N).double()
        r = res.double()
        h = (r * nw.double()) @ D.unpack_weight_fp8(*p2, 64, N).double().T \
            * torch.rsqrt(r.square().mean(1, keepdim=True) + 1e-5)
        assert (got - h).norm() < 2 ** -7 * h.norm()


@pytest.mark.parametrize("B,QH,KVH,D,longest", [
    (1, 32, 8, 64, 700), (1, 32, 8, 128, 60), (4, 32, 8, 128, 1100),
    (5, 32, 8, 128, 900), (17, 16, 1, 64, 2000), (32, 28, 4, 128, 300),
    (70, 32, 8, 128, 400), (3, 4, 4, 64, 4500)])
def test_paged_attn_step(ext, B, QH, KVH, D, longest):
    """Rotation, append and attention in one against the separate ones, at
    page edges; a row not in use leaves everything alone."""
    g = torch.Generator().manual_seed(B + longest)
    lens = torch.randint(1, longest + 1, (B,), generator=g)
    lens[:3] = torch.tensor([longest, 64, 65])[:B].clamp(max=longest)
    if B > 3:
        lens[3] = 0
    kc, vc, bt = _make_paged_kv(B, KVH, D, lens.tolist(),
                                sum(-(-n // 64) for n in lens.tolist()) + 1)
    for i, n in enumerate(lens.tolist()):         # the new token's place
        if n:
            kc[bt[i, (n - 1) // 64], :, :, (n - 1) % 64] = float("nan")
            vc[bt[i, (n - 1) // 64], :, :, (n - 1) % 64] = float("nan")
    kc2, vc2 = kc.clone(), vc.clone()
    rot = torch.rand(longest + 1, D // 2, generator=g) * 6.28
    cos, sin = rot.cos().to(dev()), rot.sin().to(dev())
    qkv = torch.randn(B, (QH + 2 * KVH) * D, generator=g).bfloat16().to(dev())
    sl = lens.int().to(dev())

    def split(t):
        q, k, v = t.split([QH * D, KVH * D, KVH * D], 1)
        return (q.view(B, QH, D), k.view(B, KVH, D), v.view(B, KVH, D))

    kept = qkv.clone()
    out = ext.paged_attn_step(*split(qkv), kc, vc, cos, sin, bt, sl,
                              D ** -0.5, False)
    assert torch.equal(qkv, kept)
    q, k, v = split(qkv)
    ext.rope_kv_append(q, k, v, kc2, vc2, cos, sin, bt, sl)
    assert torch.equal(vc, vc2)
    # products of the rotation may be fused differently: one bf16 step
    assert ((kc.float() - kc2.float()).abs()
            <= 2 ** -7 * kc2.float().abs() + 1e-6).all()
    ref = cpu_ref.paged_attn_ref(q.cpu(), kc2.cpu(), vc2.cpu(), bt.cpu(),
                                 sl.cpu(), D ** -0.5)
    torch.testing.assert_close(out.float().cpu(), ref, atol=2e-2, rtol=2e-2)
    if B <= 32:
        q, k, v = split(kept)
        step = ext.paged_attn_step(q, k, v, kc, vc, cos, sin, bt, sl,
                                   D ** -0.5, True)
        step = step.view(B, -1) if step.dim() == 3 else step
        assert torch.equal(_from_step_rows(step, B), out.view(B, -1))


# rows that read ahead: more than four, up to 64 with their key heads, none split
@pytest.mark.parametrize("lens", [
    [300, 0, 65, 64], [300, 0, 65, 1, 700],
    [5, 300, 0, 65, 1, 128, 64, 9, 0, 700, 63, 2, 90, 1000, 3, 31],
    [300, 0, 65, 1, 128, 64, 9, 10, 700, 63, 2, 90, 1000, 3, 31, 33, 17]])
@pytest.mark.parametrize("sizes", [(16,), (16 * 4097, 40), (1 << 20, 3),
                                   (25 << 20, 16), (9, 7)])
def test_paged_attn_step_reads_ahead(ext, sizes, lens):
    """What idle blocks read, ends included, changes nothing."""
    g = torch.Generator().manual_seed(len(sizes))
    B = len(lens)
    kc, vc, bt = _make_paged_kv(B, 4, 64, lens, sum(-(-n // 64) for n in lens))
    rot = torch.rand(1001, 32, generator=g)
    qkv = torch.randn(B, 24 * 64, generator=g).bfloat16().to(dev())
    q, k, v = (t.view(B, -1, 64) for t in qkv.split([1024, 256, 256], 1))
    warm = [torch.ones(n, dtype=torch.uint8, device=dev()) for n in sizes]

    def run(**more):
        return ext.paged_attn_step(
            q, k, v, kc, vc, rot.cos().to(dev()), rot.sin().to(dev()), bt,
            torch.tensor(lens, dtype=torch.int32, device=dev()), 0.125, False,
            **more)

    out = run()
    kept = kc.clone(), vc.clone()
    assert torch.equal(out, run(warm=warm))
    assert torch.equal(kept[0], kc) and torch.equal(kept[1], vc)
    assert all((w == 1).all() for w in warm)


@pytest.mark.parametrize("M", [1, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(16, 256), (48, 768), (4096, 8192)])
def test_skinny_bf16_rows(ext, M, N, K):
    torch.manual_seed(M + N)
    a = torch.randn(M, K, device=dev(), dtype=torch.bfloat16)
    w = torch.randn(N, K, device=dev(), dtype=torch.bfloat16) * K ** -0.5
    out = ext.skinny_gemm(a, ext.pack_weight_frag(w), N, K)
    want = a.double() @ w.double().T
    # exact products, f32 sums; the result is rounded to bf16
    assert (out.double() - want).norm() < 2 ** -8 * want.norm()


def test_fp8_block_sweep(ext):
    """tools/fp8_bench.py times every block shape of the probe, and each of
    them computes the product."""
    import os
    import sys
    sys.path.insert(0, os.path.join(
        os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tools"))
    import fp8_bench
    from quickstart_streaming_agents_amd.ops import dispatch as D
    torch.manual_seed(5)
    M, N, K = 24, 192, 768
    a = torch.randn(M, K, device=dev(), dtype=torch.bfloat16)
    packed = D.pack_weight_fp8(torch.randn(N, K, device=dev()).bfloat16())
    assert [t[:2] for t in fp8_bench.sweep(a, *packed, N, K)] == \
        fp8_bench.BLOCKS
    want = a.double() @ D.unpack_weight_fp8(*packed, N, K).double().T
    for waves, tiles in fp8_bench.BLOCKS:
        out = ext.skinny_gemm_fp8_probe(a, *packed, M, N, K, waves, tiles)
        assert (out.double() - want).norm() < 2 ** -8 * want.norm()
    with pytest.raises(RuntimeError, match="no such block shape"):
        ext.skinny_gemm_fp8_probe(a, *packed, M, N, K, 16, 1)


@pytest.mark.parametrize("M", [1, 4, 5, 17])
def test_embed_rows(ext, M):
    embed = torch.randn(100, 288, device=dev(), dtype=torch.bfloat16)
    w = torch.randn(288, device=dev()).bfloat16()
    tok = torch.tensor([0, 99, 7, 7, 31] * 4, device=dev())[:M]
    res, nxt, ss = ext.embed_rows(embed, tok, w)
    assert torch.equal(res, embed[tok])
    assert torch.equal(_from_step_rows(nxt, M),
                       (res.float() * w.float()).bfloat16())
    torch.testing.assert_close(ss[:M, 0], res.float().square().sum(1))


def test_llama_decode_uses_fp8_path():
    """The flagship decode path must run the fp8 kernel by default (the
    driver's native-code check: no silent bf16/rocBLAS fallback)."""
    from quickstart_streaming_agents_amd.models.llama import (LlamaConfig,
                                                              LlamaModel)
    cfg = LlamaConfig.preset("tiny")
    cfg.hidden = 256
    m = LlamaModel(cfg, device="cuda:0", seed=1)
    assert m.use_fp8
    L = m.layers[0]
    assert "wqkv_f8" in L and "wgu_f8" in L and "wdown_f8" in L
    assert m.lm_head_f8 is not None
    # numerics: one decode-shaped _linear call routes through fp8 and
    # stays close to the bf16 matmul
    x = torch.randn(8, cfg.hidden, device="cuda:0",
                    dtype=torch.bfloat16) * 0.5
    out = m._linear(x, L["wqkv"], None, L["wqkv_f8"])
    ref = x.float() @ L["wqkv"].float().T
    rel = (out.float() - ref).abs().max().item() / \
        (ref.abs().std().item() + 1e-6)
    assert rel < 0.5


def test_varlen_attention_noncausal_matches_torch():
    """Bidirectional (CAUSAL=false) varlen flash attention vs a dense
    torch reference over ragged items — the encoder's K1 attention."""
    from quickstart_streaming_agents_amd.ops import dispatch as D
    from quickstart_streaming_agents_amd.ops import ext
    torch.manual_seed(0)
    dev = "cuda:0"
    QH = KVH = 8
    Dh = 64
    lens = [37, 64, 5, 130, 1]
    n, L = len(lens), max(lens)
    ppi = (L + 63) // 64
    scale = Dh ** -0.5
    T = n * L
    q = torch.randn(T, QH, Dh, device=dev, dtype=torch.bfloat16) * 0.5
    k = torch.randn(T, KVH, Dh, device=dev, dtype=torch.bfloat16) * 0.5
    v = torch.randn(T, KVH, Dh, device=dev, dtype=torch.bfloat16) * 0.5
    kc = torch.zeros(n * ppi, KVH, Dh // 8, 64, 8, device=dev,
                     dtype=torch.bfloat16)
    vc = torch.zeros(n * ppi, KVH, Dh, 64, device=dev,
                     dtype=torch.bfloat16)
    slots = torch.arange(n * ppi * 64, dtype=torch.int32, device=dev) \
        .reshape(n, ppi * 64)[:, :L].reshape(-1).contiguous()
    D.kv_scatter(k, v, kc, vc, slots)
    bt = torch.arange(n * ppi, dtype=torch.int32, device=dev) \
        .reshape(n, ppi).contiguous()
    qb_item, qb_pos0 = [], []
    for i in range(n):
        for p0 in range(0, lens[i], 16):
            qb_item.append(i)
            qb_pos0.append(p0)
    mk = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
    for causal in (False, True):
        out = ext().paged_attn_prefill(
            q, kc, vc, bt, mk(qb_item), mk(qb_pos0),
            mk([i * L for i in range(n)]), mk([0] * n), mk(lens), scale,
            causal)
        for i in range(n):
            li = lens[i]
            qi = q[i * L:i * L + li].float()
            ki = k[i * L:i * L + li].float()
            vi = v[i * L:i * L + li].float()
            sc = torch.einsum("qhd,khd->hqk", qi, ki) * scale
            if causal:
                m = torch.triu(torch.ones(li, li, device=dev,
                                          dtype=torch.bool), 1)
                sc = sc.masked_fill(m.unsqueeze(0), float("-inf"))
            p = sc.softmax(-1)
            ref = torch.einsum("hqk,khd->qhd", p, vi).reshape(li, QH * Dh)
            got = out[i * L:i * L + li].float()
            rel = (got - ref).abs().max().item() / \
                (ref.abs().max().item() + 1e-9)
            assert rel < 2e-2, f"causal={causal} item {i}: rel {rel}"


@pytest.mark.parametrize("D,QH,KVH,rows,causal", [
    (128, 32, 8, 32, True), (128, 32, 8, 16, True), (128, 28, 4, 18, True),
    (64, 8, 8, 128, False), (64, 8, 8, 64, False), (64, 32, 8, 16, False),
    (64, 16, 1, 8, True), (128, 4, 4, 40, True)])
def test_paged_attn_prefill_blocks(ext, D, QH, KVH, rows, causal):
    """Token blocks of every shape over ragged portions with a cached prefix;
    slots that were never written hold NaN."""
    from quickstart_streaming_agents_amd.ops import dispatch as disp
    g = torch.Generator().manual_seed(D + QH + rows)
    items = [(0, 1), (63, 1), (64, 2), (5, 59), (0, 64), (100, 33), (1, 191),
             (700, 17)]
    lens = [n for _, n in items]
    np_ = [-(-(a + n) // 64) for a, n in items]
    P, cap = sum(np_), max(np_)
    kc = torch.full((P, KVH, D // 8, 64, 8), float("nan")).bfloat16().to(dev())
    vc = torch.full((P, KVH, D, 64), float("nan")).bfloat16().to(dev())
    pages = torch.randperm(P, generator=g).int()
    bt = torch.zeros(len(items), cap, dtype=torch.int32)
    T = sum(lens)
    q = torch.randn(T, QH, D, generator=g).bfloat16().to(dev())
    kv, at, offs = [], 0, []
    for i, (a, n) in enumerate(items):
        bt[i, :np_[i]] = pages[at:at + np_[i]]
        at += np_[i]
        offs.append(sum(lens[:i]))
        k = torch.randn(a + n, KVH, D, generator=g).bfloat16().to(dev())
        v = torch.randn(a + n, KVH, D, generator=g).bfloat16().to(dev())
        pos = torch.arange(a + n)
        slots = (bt[i][pos // 64] * 64 + pos % 64).int().to(dev())
        disp.kv_scatter(k, v, kc, vc, slots)
        kv.append((k.double(), v.double()))
    blocks = [(i, p) for i, n in enumerate(lens) for p in range(0, n, rows)]
    mk = lambda x: torch.tensor(x, dtype=torch.int32, device=dev())
    out = ext.paged_attn_prefill(
        q, kc, vc, bt.to(dev()), mk([b[0] for b in blocks]),
        mk([b[1] for b in blocks]), mk(offs), mk([a for a, _ in items]),
        mk(lens), D ** -0.5, causal, rows)
    R = QH // KVH
    for i, (a, n) in enumerate(items):
        k, v = (t.repeat_interleave(R, 1).transpose(0, 1) for t in kv[i])
        qi = q[offs[i]:offs[i] + n].double().transpose(0, 1)
        s = qi @ k.transpose(1, 2).contiguous() * D ** -0.5
        if causal:
            j = torch.arange(a + n, device=dev())
            s = s.masked_fill(j[None] > j[a:, None], float("-inf"))
        ref = (s.softmax(-1) @ v).transpose(0, 1).reshape(n, QH * D)
        got = out[offs[i]:offs[i] + n].double()
        # probabilities and the result are rounded to bf16: 2^-9 each of
        # values up to the largest |v|, and independent over the keys
        assert (got - ref).norm() <= 5e-3 * ref.norm(), i
        assert (got - ref).abs().max() <= 2 ** -7 * v.abs().max(), i


@pytest.mark.parametrize("D,QH,KVH,rows,scale", [
    (128, 8, 2, 32, 1.0), (64, 8, 2, 32, 1.0), (128, 8, 2, 16, -1.0),
    (64, 4, 4, 64, 1.0)])
def test_paged_attn_prefill_turns(ext, D, QH, KVH, rows, scale):
    """Every number of pages up to five, waves of a block that end a page
    apart, larger scores on later pages, and keys of NaN on any page but the
    first one, which count as none."""
    from quickstart_streaming_agents_amd.ops import dispatch as disp
    g = torch.Generator().manual_seed(D + rows)
    R = QH // KVH
    items = [(a + d, n) for a in (0, 64, 128, 192) for d, n in
             ((0, 1), (0, 64), (33, 32), (50, 31), (63, 2), (47, 80))]
    lens = [n for _, n in items]
    np_ = [-(-(a + n) // 64) for a, n in items]
    kc = torch.full((sum(np_), KVH, D // 8, 64, 8), float("nan"))
    kc = kc.bfloat16().to(dev())
    vc = torch.full((sum(np_), KVH, D, 64), float("nan")).bfloat16().to(dev())
    bt = torch.zeros(len(items), max(np_), dtype=torch.int32)
    offs = [sum(lens[:i]) for i in range(len(items))]
    q = torch.randn(sum(lens), QH, D, generator=g).bfloat16().to(dev())
    kv, at = [], 0
    for i, (a, n) in enumerate(items):
        bt[i, :np_[i]] = torch.arange(at, at + np_[i])
        at += np_[i]
        k = torch.randn(a + n, KVH, D, generator=g)
        k = k * (1 + torch.arange(a + n) / 64).floor()[:, None, None]
        for j in (70, 129, 200):
            k[j:j + 1] = float("nan")
        k, v = (t.bfloat16().to(dev()) for t in (
            k, torch.randn(a + n, KVH, D, generator=g)))
        pos = torch.arange(a + n)
        disp.kv_scatter(k, v, kc, vc,
                        (bt[i][pos // 64] * 64 + pos % 64).int().to(dev()))
        kv.append((k.double(), v.double()))
    blocks = [(i, p) for i, n in enumerate(lens) for p in range(0, n, rows)]
    mk = lambda x: torch.tensor(x, dtype=torch.int32, device=dev())
    out = ext.paged_attn_prefill(
        q, kc, vc, bt.to(dev()), mk([b[0] for b in blocks]),
        mk([b[1] for b in blocks]), mk(offs), mk([a for a, _ in items]),
        mk(lens), scale * D ** -0.5, True, rows)
    for i, (a, n) in enumerate(items):
        k, v = (t.repeat_interleave(R, 1).transpose(0, 1) for t in kv[i])
        qi = q[offs[i]:offs[i] + n].double().transpose(0, 1)
        s = qi @ k.transpose(1, 2).contiguous() * (scale * D ** -0.5)
        j = torch.arange(a + n, device=dev())
        s = s.masked_fill(s.isnan() | (j[None] > j[a:, None]), float("-inf"))
        ref = (s.softmax(-1) @ v).transpose(0, 1).reshape(n, QH * D)
        got = out[offs[i]:offs[i] + n].double()
        # as above: weights and results rounded to bf16
        assert (got - ref).norm() <= 5e-3 * ref.norm(), (i, a, n)
        assert (got - ref).abs().max() <= 2 ** -7 * v.abs().max(), (i, a, n)


@pytest.mark.parametrize("T,QH,KVH,D", [
    (1, 8, 8, 64), (63, 4, 2, 128), (65, 32, 8, 128), (200, 28, 4, 128),
    (130, 16, 1, 64)])
def test_rope_kv_scatter(ext, T, QH, KVH, D):
    """One pass against rotation and scatter apart; tokens in any slots."""
    g = torch.Generator().manual_seed(T + D)
    P = T // 64 + 3
    kc = torch.randn(P, KVH, D // 8, 64, 8, generator=g).bfloat16().to(dev())
    vc = torch.randn(P, KVH, D, 64, generator=g).bfloat16().to(dev())
    kc2, vc2 = kc.clone(), vc.clone()
    slots = torch.randperm(P * 64, generator=g)[:T].int().to(dev())
    pos = torch.randint(0, 500, (T,), generator=g).int().to(dev())
    rot = torch.rand(500, D // 2, generator=g) * 6.28
    cos, sin = rot.cos().to(dev()), rot.sin().to(dev())
    qkv = torch.randn(T, (QH + 2 * KVH) * D, generator=g).bfloat16().to(dev())
    twin = qkv.clone()

    def split(t):
        q, k, v = t.split([QH * D, KVH * D, KVH * D], 1)
        return (q.view(T, QH, D), k.view(T, KVH, D), v.view(T, KVH, D))

    q, k, v = split(qkv)
    ext.rope_kv_scatter(q, k, v, kc, vc, cos, sin, pos, slots)
    q2, k2, v2 = split(twin)
    ext.rope_inplace(q2, k2, cos, sin, pos)
    ext.kv_scatter(k2, v2, kc2, vc2, slots)
    assert torch.equal(vc, vc2)
    # products of the rotation may be fused differently: one bf16 step
    for a, b in ((q, q2), (kc, kc2)):
        assert ((a.float() - b.float()).abs()
                <= 2 ** -7 * b.float().abs() + 1e-6).all()


@pytest.mark.parametrize("D,QH,KVH,rows,scale", [
    (128, 32, 8, 32, 1.0), (128, 28, 4, 9, 1.0), (64, 8, 8, 128, -1.0),
    (64, 16, 1, 4, 1.0)])
def test_prefill_rotates_queries(ext, D, QH, KVH, rows, scale):
    """Queries turned on their way into the attention, at the position of each
    row, against the same turned before."""
    g = torch.Generator().manual_seed(D + rows)
    items = [(0, 1), (63, 2), (5, 130), (64, 64), (200, 33)]
    lens = [n for _, n in items]
    np_ = [-(-(a + n) // 64) for a, n in items]
    bt = torch.zeros(len(items), max(np_), dtype=torch.int32)
    for i, n in enumerate(np_):
        bt[i, :n] = torch.arange(sum(np_[:i]), sum(np_[:i]) + n)
    T, P = sum(lens), sum(np_)
    qkv = torch.randn(T, (QH + 2 * KVH) * D, generator=g).bfloat16().to(dev())
    twin = qkv.clone()
    rot = torch.rand(233, D // 2, generator=g) * 6.28    # up to the last position
    cos, sin = rot.cos().to(dev()), rot.sin().to(dev())
    mk = lambda x: torch.tensor(x, dtype=torch.int32, device=dev())
    pos = mk([a + i for a, n in items for i in range(n)])
    slots = mk([int(bt[i, p // 64]) * 64 + p % 64
                for i, (a, n) in enumerate(items) for p in range(a, a + n)])
    blocks = [(i, p) for i, n in enumerate(lens) for p in range(0, n, rows)]
    maps = (bt.to(dev()), mk([b[0] for b in blocks]),
            mk([b[1] for b in blocks]), mk(list(np.cumsum(lens) - lens)),
            mk([a for a, _ in items]), mk(lens), scale * D ** -0.5, True, rows)
    kc = torch.randn(P, KVH, D // 8, 64, 8, generator=g).bfloat16().to(dev())
    vc = torch.randn(P, KVH, D, 64, generator=g).bfloat16().to(dev())
    kc2, vc2 = kc.clone(), vc.clone()

    def split(t):
        return [x.view(T, -1, D) for x in
                t.split([QH * D, KVH * D, KVH * D], 1)]

    q, k, v = split(qkv)
    ext.rope_kv_scatter(q, k, v, kc, vc, cos, sin, pos, slots, turn_q=False)
    assert torch.equal(qkv, twin)                        # nothing of it changed
    got = ext.paged_attn_prefill(q, kc, vc, *maps, cos, sin)
    q2, k2, v2 = split(twin)
    ext.rope_kv_scatter(q2, k2, v2, kc2, vc2, cos, sin, pos, slots)
    assert torch.equal(kc, kc2) and torch.equal(vc, vc2)
    # the same sums of the same products: no bit of it differs
    assert torch.equal(got, ext.paged_attn_prefill(q2, kc2, vc2, *maps))


def test_prefill_refuses_host_angles(ext):
    """Rotation tables whose memory is the host's are an error, not a launch."""
    mk = lambda *x: torch.tensor(x, dtype=torch.int32, device=dev())
    q = torch.randn(5, 4, 64).bfloat16().to(dev())
    kc = torch.randn(1, 1, 8, 64, 8).bfloat16().to(dev())
    vc = torch.randn(1, 1, 64, 64).bfloat16().to(dev())
    args = (q, kc, vc, mk(0).view(1, 1), mk(0), mk(0), mk(0), mk(0), mk(5),
            0.125, True, 16)
    t = torch.ones(64, 32)
    assert torch.isfinite(
        ext.paged_attn_prefill(*args, t.to(dev()), t.to(dev()))).all()
    for angles in ((t, t.to(dev())), (t.to(dev()), t)):
        with pytest.raises(RuntimeError, match="must be where q is"):
            ext.paged_attn_prefill(*args, *angles)


@pytest.mark.parametrize("D,H", [(64, 8), (128, 4)])
@pytest.mark.parametrize("lens", [[1], [64, 63, 65, 1, 130], [512, 3, 128]])
def test_encoder_attn(ext, lens, D, H):
    """Rows of q, k and v as the projection leaves them, items at tile edges,
    blocks in any order; weights and results are rounded to bf16."""
    g = torch.Generator().manual_seed(D + len(lens))
    T, A = sum(lens), H * D
    qkv = torch.randn(T, 3 * A, generator=g).bfloat16()
    rot = torch.rand(512, D // 2, generator=g, dtype=torch.float64) * 6.28
    cos, sin = rot.cos().float(), rot.sin().float()
    off = np.cumsum(lens) - lens
    blocks = [(i, t) for i, n in enumerate(lens) for t in range(0, n, 64)][::-1]
    got = ext.encoder_attn(
        qkv.to(dev()), cos.to(dev()), sin.to(dev()),
        *(torch.tensor(x, dtype=torch.int32, device=dev())
          for x in ([b[0] for b in blocks], [b[1] for b in blocks],
                    off.tolist(), lens)), H, D ** -0.5).cpu().double()

    def rotated(x, n):
        a, b = x.float().chunk(2, -1)
        c, s = cos[:n, None], sin[:n, None]
        return torch.cat([a * c - b * s, a * s + b * c], -1).bfloat16() \
            .double()

    for o, n in zip(off, lens):
        q, k, v = qkv[o:o + n].view(n, 3, H, D).unbind(1)
        p = torch.einsum("ihd,jhd->hij", rotated(q, n), rotated(k, n))
        p = (p * D ** -0.5).softmax(-1)
        want = torch.einsum("hij,jhd->ihd", p, v.double()).reshape(n, A)
        # of the weights 2**-9, of the result 2**-9, of a rotated number
        # rounded the other way 2**-8 of some score of a few units
        scale = torch.einsum("hij,jhd->ihd", p, v.double().abs()).reshape(n, A)
        assert ((got[o:o + n] - want).abs() <= 2 ** -6 * scale + 1e-6).all()


def test_encoder_attn_nan_scores(ext):
    """A NaN score counts as no key, in whole tiles and in the last one, as in
    the paged kernel; a row that sees nothing else comes out as zero."""
    g = torch.Generator().manual_seed(4)
    H, D, lens, bad = 4, 64, [1, 150], (0, 1 + 10, 1 + 70, 1 + 149)
    T = sum(lens)
    qkv = torch.randn(T, 3, H, D, generator=g).bfloat16()
    qkv[list(bad), 1, 2] = float("nan")
    still = torch.ones(200, D // 2), torch.zeros(200, D // 2)
    mk = lambda *x: torch.tensor(x, dtype=torch.int32, device=dev())
    got = ext.encoder_attn(
        qkv.view(T, -1).to(dev()), still[0].to(dev()), still[1].to(dev()),
        mk(0, 1, 1, 1), mk(0, 0, 64, 128), mk(0, 1), mk(*lens), H,
        D ** -0.5).cpu().double().view(T, H, D)
    assert not got[0, 2].any()
    q, k, v = qkv[1:].double().unbind(1)
    s = torch.einsum("ihd,jhd->hij", q, k) * D ** -0.5
    p = s.masked_fill(s.isnan(), float("-inf")).softmax(-1)
    want = torch.einsum("hij,jhd->ihd", p, v)
    scale = torch.einsum("hij,jhd->ihd", p, v.abs())
    # weights and the result are rounded to bf16: 2**-9 each
    assert ((got[1:] - want).abs() <= 2 ** -7 * scale + 1e-6).all()


@pytest.mark.parametrize("M", [1, 33, 65, 1000, 5600])
@pytest.mark.parametrize("N,K,glu", [
    (32, 64, False), (1536, 384, False), (400, 512, False), (96, 1536, False),
    (3072, 384, True), (96, 192, True)])
def test_short_gemm(ext, M, N, K, glu):
    """Every tile shape, ragged ends of rows and columns, rows of a slice.  An
    f32 sum of K products and a rounding to bf16; the activation's slope is
    1.1 at most."""
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K + 16, generator=g).bfloat16().to(dev())[:, 8:K + 8]
    w = torch.randn(N, K, generator=g).mul(K ** -0.5).bfloat16().to(dev())
    got = ext.short_gemm(x, w, glu).double()
    a, b = x.double(), w.double()
    want, err = a @ b.T, K * 2.0 ** -24 * (a.abs() @ b.abs().T)
    if glu:
        z, u = want.chunk(2, 1)
        want = torch.nn.functional.silu(z) * u
        err = 1.1 * err[:, :N // 2] * u.abs() + z.abs() * err[:, N // 2:] + \
            2.0 ** -20 * want.abs()
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + err + 1e-30).all()


@pytest.mark.parametrize("M,N,glu", [(33, 3072, True), (1000, 400, False)])
@pytest.mark.parametrize("steps", [1, 2, 3, 7, 8, 9, 10, 11, 12, 13, 14, 24])
def test_short_gemm_steps(ext, M, N, glu, steps):
    """The tiles of 32 x 64, up to eight steps with one ahead, beyond with every
    number of them behind the last six that are under way together."""
    assert -(-M // 32) * (N // (32 if glu else 16)) > (128 if glu else 256)
    assert -(-M // 64) * -(-N // 64) < 128
    test_short_gemm(ext, M, N, 64 * steps, glu)


@pytest.mark.parametrize("M,N,K,glu", [
    (1, 32, 64, False), (32, 384, 1536, False), (40, 96, 1088, False),
    (17, 48, 576, False), (250, 512, 1600, False), (31, 64, 2112, True),
    (33, 1536, 448, True), (5, 32, 512, True)])
def test_short_gemm_few_rows(ext, M, N, K, glu):
    """K in shares of eight waves: fewer steps than waves, remainders of the steps
    that are under way together, ragged rows.  The bound is that of the tiles."""
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K + 8, generator=g).bfloat16().to(dev())[:, :K]
    w = torch.randn(N, K, generator=g).mul(K ** -0.5).bfloat16().to(dev())
    got = ext.short_gemm(x, w, glu).double()
    a, b = x.double(), w.double()
    want, err = a @ b.T, K * 2.0 ** -24 * (a.abs() @ b.abs().T)
    if glu:
        z, u = want.chunk(2, 1)
        want = torch.nn.functional.silu(z) * u
        err = 1.1 * err[:, :N // 2] * u.abs() + z.abs() * err[:, N // 2:] + \
            2.0 ** -20 * want.abs()
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + err + 1e-30).all()


@pytest.mark.parametrize("M", [3, 700])
def test_gates_far_from_zero(ext, M):
    """Gates whose 1 + e^-z is beyond 2^126, the largest number with a normal
    reciprocal, in every kernel that applies one to numbers given to it: the
    quotient is a normal number and comes out as one."""
    from quickstart_streaming_agents_amd.ops import dispatch as D
    from quickstart_streaming_agents_amd.ops import lm_ext
    N, K = 256, 512
    z = torch.tensor([-87.0, -87.5, -88.0, -88.5]).repeat(N // 4).bfloat16()
    up = torch.full((N,), 2.0 ** 100).bfloat16()
    silu = z.double() / (1 + torch.exp(-z.double()))
    want = (silu * up.double()).expand(M, N)

    def close(got, want=want):
        # the exponential's argument times log2(e), rounded: 2^-17 at 88; the
        # factor and the result rounded to bf16
        err = (got.cpu().double() - want).abs()
        assert (err <= 2.0 ** -8 * want.abs()).all()

    rows = [t.expand(M, N).contiguous().to(dev()) for t in (z, up)]
    close(ext.swiglu(*rows))
    close(D.glu(*rows))
    # products: the first column of W is the gate's and the factor's row
    x = torch.zeros(M, K).bfloat16()
    x[:, 0] = 1
    w = torch.zeros(2 * N, K).bfloat16()
    w[:, 0] = torch.cat((z, up))
    x, w = x.to(dev()), w.to(dev())
    close(ext.short_gemm(x, w, True))
    close(lm_ext().rows_glu(x, w, False, False))
    close(lm_ext().wide_gemm(x, w, 0, 3))
    # a convolution of one tap: the result itself is as small
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device=dev())
    y = D.conv_silu(rows[0], torch.ones(1, N, device=dev()),
                    torch.zeros(N, device=dev()),
                    torch.zeros(M, 0, N, device=dev()).bfloat16(), None, None,
                    None, i32(*[5] * M), None, i32(*range(M)))
    close(y, silu.expand(M, N))


def test_mean_rows(ext):
    lens = [1, 3, 4, 5, 700]
    x = torch.randn(sum(lens), 520, device=dev()).bfloat16()
    off = np.cumsum(lens) - lens
    got = ext.mean_rows(x, torch.tensor(off, dtype=torch.int32, device=dev()),
                        torch.tensor(lens, dtype=torch.int32, device=dev()))
    want = torch.stack([x[o:o + n].double().mean(0)
                        for o, n in zip(off, lens)])
    # f32 sums of up to 175 values in four parts
    torch.testing.assert_close(got.double(), want, rtol=1e-5, atol=1e-6)


def test_hash_join_gpu_matches_cpu_semantics():
    """K8 hash build/probe on GPU vs the CPU dispatch fallback: random
    keys with duplicates, latest-event-time-wins, TTL cutoff."""
    from quickstart_streaming_agents_amd.ops import dispatch as D
    torch.manual_seed(11)
    N, M = 5000, 3000
    keys = torch.randint(0, 1500, (N,), dtype=torch.int64)  # many dups
    ts = torch.randint(0, 1_000_000, (N,), dtype=torch.int64)
    probe = torch.randint(0, 2000, (M,), dtype=torch.int64)  # some misses
    cutoff = 400_000
    cpu_table = D.hash_build(keys, ts)
    cpu_rows = D.hash_probe(cpu_table, probe, cutoff)
    gpu_table = D.hash_build(keys.cuda(), ts.cuda())
    gpu_rows = D.hash_probe(gpu_table, probe.cuda(), cutoff).cpu()
    assert torch.equal(cpu_rows, gpu_rows)
    # spot-check semantics: row returned is the max-(ts, idx) for its key
    for i in range(0, M, 137):
        r = int(cpu_rows[i])
        k = int(probe[i])
        cands = [(int(ts[j]), j) for j in range(N) if int(keys[j]) == k]
        if not cands:
            assert r == -1
            continue
        best_ts, best_j = max(cands)
        if best_ts >= cutoff:
            assert r == best_j
        else:
            assert r == -1


def test_lab1_gpu_join_pipeline_matches_cpu():
    """lab1 enriched_orders through the GPU hash-join kernels == CPU."""
    from quickstart_streaming_agents_amd.labs import datagen, pipelines
    from quickstart_streaming_agents_amd.wire import Broker
    b1, b2 = Broker(), Broker()
    datagen.publish_lab1(b1)
    datagen.publish_lab1(b2)
    cpu = pipelines.lab1_enriched_orders(b1, use_gpu=False)
    gpu = pipelines.lab1_enriched_orders(b2, use_gpu=True)
    assert cpu == gpu and len(cpu) >= 1


def test_gemm_fp8_batch_matches_dequant_ref():
    """Batched-M fp8 weight-stream GEMM (LDS-staged A, optional split-K)
    vs the dequantized fp32 reference, across the llama decode shapes and
    ragged M values."""
    from quickstart_streaming_agents_amd.ops import dispatch as D
    from quickstart_streaming_agents_amd.ops import ext
    torch.manual_seed(7)
    cases = [
        (192, 6144, 4096, 4),    # qkv at bench batch (split-K)
        (192, 4096, 4096, 4),    # wo
        (192, 28672, 4096, 1),   # wgu
        (192, 4096, 14336, 4),   # wdown
        (33, 4096, 4096, 2),     # just past the skinny cutover
        (256, 1024, 1024, 1),    # full M tile
        (100, 2048, 512, 2),     # ragged M, small K
    ]
    for M, N, K, splitk in cases:
        a = torch.randn(M, K, device="cuda:0", dtype=torch.bfloat16) * 0.5
        w = torch.randn(N, K, device="cuda:0", dtype=torch.bfloat16) * 0.02
        qf, s = D.pack_weight_fp8(w)
        out = ext().gemm_fp8_batch(a, qf, s, N, K, splitk)
        wd = D.unpack_weight_fp8(qf, s, N, K)
        ref = a.float() @ wd.T
        err = (out.float() - ref).abs().max().item()
        rel = err / (ref.abs().max().item() + 1e-6)
        assert rel < 2e-2, f"M{M} N{N} K{K} sk{splitk}: rel {rel}"


def test_llama_batched_decode_routes_fp8():
    """_linear at decode-batch M routes through the batched fp8 kernel
    and matches the bf16 matmul within quantization error."""
    from quickstart_streaming_agents_amd.models.llama import (LlamaConfig,
                                                              LlamaModel)
    cfg = LlamaConfig.preset("tiny")
    m = LlamaModel(cfg, device="cuda:0", seed=2)
    L = m.layers[0]
    x = torch.randn(192, cfg.hidden, device="cuda:0",
                    dtype=torch.bfloat16) * 0.5
    out = m._linear(x, L["wgu"], None, L["wgu_f8"])
    ref = x.float() @ L["wgu"].float().T
    rel = (out.float() - ref).abs().max().item() / \
        (ref.abs().std().item() + 1e-6)
    assert rel < 0.5


@pytest.mark.parametrize("fuse", [False, True])
def test_paged_attn_without_pages(ext, fuse):
    """No rows, a table without columns, one without the last, empty rows."""
    B, QH, KVH, D = 5, 8, 4, 64
    kc, vc, bt = _make_paged_kv(B, KVH, D, [70, 3, 1, 0, 0], 5)
    kept = kc.clone(), vc.clone()
    qkv = torch.randn(B, (QH + 2 * KVH) * D, device=dev()).bfloat16()
    rot = torch.rand(128, D // 2, device=dev())

    def run(rows, table, lens):
        q, k, v = (t.view(B, -1, D)[:rows] for t in
                   qkv.split([QH * D, KVH * D, KVH * D], 1))
        sl = torch.tensor(lens, dtype=torch.int32, device=dev())
        if not fuse:
            return ext.paged_attn_decode(q, kc, vc, table, sl, 0.125)
        return ext.paged_attn_step(q, k, v, kc, vc, rot, rot, table, sl,
                                   0.125, False)

    assert run(0, bt[:0], []).shape == (0, QH, D)
    assert run(0, bt[:0, :1].expand(0, 40).contiguous(), []).numel() == 0
    none = run(B, bt[:, :0].contiguous(), [0] * B)
    assert none.shape == (B, QH, D) and not none.any()
    assert torch.equal(kc, kept[0]) and torch.equal(vc, kept[1])
    want = run(B, bt, [70, 3, 1, 0, 0])
    assert torch.equal(run(B, bt[:3].contiguous(), [70, 3, 1, 0, 0]), want)
    assert want[:3].any() and not want[3:].any()
