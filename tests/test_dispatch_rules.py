"""Which form of a kernel a call takes: rules of sizes alone, on the host."""

from __future__ import annotations

import pytest
import torch

from quickstart_streaming_agents_amd.ops import (
    ext, have_ext, have_lm_ext, lm_ext)

pytestmark = pytest.mark.skipif(not (have_ext() and have_lm_ext()),
                                reason="extensions not built")


@pytest.mark.parametrize("pages", [0, 1, 16, 17, 40])
def test_decode_attention_of_no_rows(pages):
    """A batch without rows has no blocks to share its pages."""
    assert ext().paged_attn_split(0, 32, 8, pages, 128)[1] == 1


# rows, key heads, pages: either side of every line of the rule, tables that a
# block of eight waves walks once, twice and often
SPLITS = [(12, 4, 4), (12, 4, 5), (12, 4, 16), (12, 4, 17), (7, 7, 16),
          (7, 7, 17), (8, 8, 33), (13, 5, 16), (13, 5, 17), (13, 5, 40),
          (16, 8, 17), (16, 8, 33), (43, 3, 16), (43, 3, 17), (43, 3, 33),
          (32, 8, 4), (32, 8, 17), (32, 8, 40), (257, 1, 32), (257, 1, 33),
          (257, 1, 50), (383, 1, 33), (48, 8, 33), (1, 1, 70), (1, 8, 130),
          (5, 1, 17), (3, 2, 64)]


def _kind(pairs, pages, heads=1):
    """Waves and blocks; of few rows any number of blocks, as 2."""
    waves, blocks = ext().paged_attn_split(pairs // heads, 2 * heads, heads,
                                           pages, 128)
    return waves, min(blocks, 2) if pairs <= 48 else blocks


def test_sizes_reach_every_split():
    want = {_kind(pairs, pages) for pairs in range(1, 520)
            for pages in range(1, 200)}
    assert len(want) == 6
    assert {_kind(b * g, n, g) for b, g, n in SPLITS} == want


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("rows,heads,pages", SPLITS)
def test_decode_attention_splits(rows, heads, pages, D):
    """Lengths of no key, one, ends of pages, fewer pages than a row has waves
    and the whole table, whose other columns point anywhere."""
    g = torch.Generator().manual_seed(rows + pages)
    R, top = 3, pages * 64
    lens = torch.randint(1, top + 1, (rows,), generator=g)
    some = [top, 0, 1, 64, 65, top - 63, 5 * 64, 9 * 64 + 1, top - 64]
    lens[:len(some)] = torch.tensor(some)[:rows].clamp(0, top)
    used = [-(-int(n) // 64) for n in lens]
    total = sum(used) + 1
    table = torch.randint(0, total, (rows, pages), generator=g,
                          dtype=torch.int32)
    order, at = torch.randperm(total, generator=g).int(), 0
    for i, n in enumerate(used):
        table[i, :n] = order[at:at + n]
        at += n
    dev, bf = "cuda:0", torch.bfloat16

    def rnd(*s):
        return torch.randn(*s, device=dev, dtype=bf)

    torch.manual_seed(pages)
    kc, vc = rnd(total, heads, D // 8, 64, 8), rnd(total, heads, D, 64)
    qkv = rnd(rows, (R + 2) * heads * D)
    q, k, v = (t.view(rows, -1, D) for t in qkv.split(
        [R * heads * D, heads * D, heads * D], 1))
    rot = torch.rand(top, D // 2, device=dev) * 6.28
    cos, sin = rot.cos(), rot.sin()
    bt, sl = table.to(dev), lens.int().to(dev)

    def check(out, q):
        for i, n in enumerate(lens.tolist()):
            if n == 0:
                assert not out[i].any()
                continue
            p = bt[i, :used[i]].long()
            ks = kc[p].permute(1, 0, 3, 2, 4).reshape(heads, -1, D)[:, :n]
            vs = vc[p].permute(1, 0, 3, 2).reshape(heads, -1, D)[:, :n]
            qs = q[i].view(heads, R, D).float()
            s = torch.matmul(qs, ks.float().transpose(1, 2).contiguous())
            ref = torch.matmul((s * D ** -0.5).softmax(-1), vs.float())
            err = out[i].view(heads, R, D).float() - ref
            # probabilities and the result are rounded to bf16, 2^-9 each
            assert err.norm() <= 5e-3 * ref.norm(), (i, n)
            assert err.abs().max() <= 2 ** -7 * vs.abs().max(), (i, n)

    # the step first: it writes the new keys and values that both attend to
    out = ext().paged_attn_step(q, k, v, kc, vc, cos, sin, bt, sl, D ** -0.5,
                                False)
    live = sl > 0
    pos = (sl - 1).clamp(min=0)
    turned = q.clone()
    ext().rope_inplace(turned, k.clone(), cos, sin, pos)
    check(out, turned)
    i = live.nonzero()[:, 0]
    slot = bt[i, (pos[i] // 64).long()].long(), (pos[i] % 64).long()
    assert torch.equal(vc[slot[0], :, :, slot[1]], v[i])
    check(ext().paged_attn_decode(turned, kc, vc, bt, sl, D ** -0.5), turned)


@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("K", [2304, 3072, 4096, 8192])
def test_tiles_of_the_fp8_stream(K, glu):
    """9 to 16 rows: four tiles a block where no CU gets more of them than in blocks
    of two, and from 24577 columns on."""
    def tiles(M, N, k=K):
        return ext().skinny_gemm_fp8_block(M, N, k, glu, False)[1]

    for M in (9, 16):
        for N in (24_704, 28_672, 32_768, 41_088, 45_056, 49_152, 57_472, 65_536,
                  131_072):
            assert tiles(M, N) == 4, N
        for N in (18_432, 24_576, 32_896, 36_864, 40_960, 49_280, 57_344):
            assert tiles(M, N) == 2, N
            assert tiles(M, N + 4096, 2048) == 2
    for N in range(16_512, 131_072, 1664):
        assert tiles(17, N) == tiles(32, N) == 4
        assert tiles(8, N) == (2 if glu or N < 65_536 else 4)


@pytest.mark.parametrize("M,N,K,block", [
    (9, 12_288, 2048, (8, 4)), (16, 16_384, 3072, (8, 4)), (16, 14_336, 3328, (8, 2)),
    (24, 12_288, 1024, (8, 4)), (24, 15_360, 4096, (8, 4)), (24, 16_384, 4096, (4, 4)),
    (24, 16_384, 8192, (8, 4)), (8, 14_336, 2048, (8, 2)), (24, 12_160, 2048, (8, 2)),
    (16, 16_400, 4096, (8, 1)), (3, 4096, 2048, (4, 1)), (3, 4096, 2304, (8, 1))])
def test_blocks_of_the_fp8_stream(M, N, K, block):
    assert ext().skinny_gemm_fp8_block(M, N, K, False, False) == block
    if N >= 12_288 and N % 32 == 0:
        assert ext().skinny_gemm_fp8_block(M, N, K, False, True) == (8, 2)


@pytest.mark.parametrize("M,N,K", [
    (64, 12288, 8192), (64, 12288, 4096), (64, 16384, 2048), (33, 16384, 12288),
    (48, 14336, 4096), (64, 9216, 4096), (128, 8192, 4096)])
def test_few_rows_of_many_columns_take_wider_tiles(M, N, K):
    """Tiles of 64 x 32 cost up to half as much again here."""
    assert lm_ext().rows_gemm_plan(M, N, K, False)[0] != 0


@pytest.mark.parametrize("M,N,K", [(33, 2048, 2048), (64, 2048, 4096),
                                   (192, 1024, 512)])
def test_smallest_tiles_where_they_are_few(M, N, K):
    assert lm_ext().rows_gemm_plan(M, N, K, False)[0] == 0


@pytest.mark.parametrize("M,N,K,inside", [
    (33, 2048, 16384, False), (64, 4096, 8192, False), (100, 1024, 4096, False),
    (64, 16384, 2048, True), (192, 28672, 4096, True), (100, 4096, 2048, True),
    (1024, 28672, 4096, True), (13_800, 16384, 2048, True),
    (8800, 3072, 384, True), (9000, 28672, 4096, False)])
def test_gated_products_that_would_split_k(M, N, K, inside):
    """The activation inside a product leaves K whole."""
    assert lm_ext().rows_gemm_sizes(M, N, K, True) == inside
    _, shares = lm_ext().rows_gemm_plan(M, N, K, False)
    assert inside or shares > 1 or not lm_ext().rows_gemm_sizes(M, N, K, False)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(33, 2048, 4096), (100, 1024, 4096),
                                   (100, 4096, 2048)])
def test_gated_layers_on_either_side(M, N, K):
    """Inside or apart, gate and up are rounded before the activation."""
    from quickstart_streaming_agents_amd.models.layers import DenseGLU
    from quickstart_streaming_agents_amd.ops import dispatch as D
    torch.manual_seed(M + K)
    dev, bf = "cuda:0", torch.bfloat16
    gate, up = (torch.randn(N // 2, K, device=dev, dtype=bf) * K ** -0.5
                for _ in range(2))
    x = torch.randn(M, K, device=dev, dtype=bf)
    ff = DenseGLU(gate, up, torch.eye(N // 2, device=dev, dtype=bf))
    assert D.glu_linear_ok(x, ff.gate_up.w) == \
        lm_ext().rows_gemm_sizes(M, N, K, True)
    a, b = x.double(), ff.gate_up.w.double()
    g, u = (a @ b.T).chunk(2, 1)
    # gate and up: f32 sums of K products, __expf and a rounding to bf16 each;
    # the activation's slope is 1.13 at most, the result is rounded
    e = K * 2.0 ** -24 * (a.abs() @ b.abs().T) + 2.0 ** -20 \
        + 2.0 ** -8 * (a @ b.T).abs()
    (eg, eu), f = e.chunk(2, 1), torch.nn.functional.silu(g)
    want = f * u
    bound = (2.0 ** -8 + 2.0 ** -18) * want.abs() + 1.13 * eg * u.abs() \
        + (f.abs() + eg) * eu
    got = ff.gate_up.glu(x, "silu").double()
    assert ((got - want).abs() <= bound).all()


@pytest.mark.parametrize("n,k,rows", [
    (6144, 3072, 33), (8192, 2304, 33), (6144, 2048, 17), (5632, 3072, 17),
    (10240, 2048, 17), (2048, 4096, 17), (4096, 2048, 33)])
def test_rows_at_which_a_layer_leaves_the_packed_stream(n, k, rows):
    from quickstart_streaming_agents_amd.models.layers import Linear
    assert Linear(torch.empty(n, k, device="meta")).rows == rows
