"""Products of many rows (ops/hip/wide_gemm.hip): every tile at the ends of rows,
columns and K, blocks that take several tiles, and the split of a product's rows."""

import pytest
import torch

from quickstart_streaming_agents_amd.ops import dispatch as D
from quickstart_streaming_agents_amd.ops import lm_ext

BF, DEV = torch.bfloat16, "cuda:0"
TILES = [(256, 256, 2), (192, 256, 2), (256, 192, 2), (192, 192, 2),
         (256, 128, 3), (128, 256, 2), (192, 128, 3), (128, 192, 3),
         (128, 128, 4)]            # rows, columns, stages ahead


def operands(M, N, K, scale=1.0):
    """Rows of a slice, 16 bytes aligned."""
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K + 24, generator=g).to(BF).to(DEV)[:, 8:K + 8]
    w = (torch.randn(N, K, generator=g) * scale).to(BF).to(DEV)
    torch.full((M, N), float("nan"), dtype=BF, device=DEV)      # stale memory
    return x, w


def check(got, x, w, act):
    """f32 sums of K products; gate and up are rounded to bf16 (but for act 3)
    before an activation whose slope is at most 1.13 and whose __expf and division
    are good to 2^-20; the result is rounded to bf16."""
    a, b, K = x.double(), w.double(), x.shape[1]
    y, e = a @ b.T, K * 2.0 ** -24 * (a.abs() @ b.abs().T)
    if act == 0:
        assert ((got.double() - y).abs() <= 2.0 ** -8 * y.abs() + e).all()
        return
    e = e + 2.0 ** -20 + (0.0 if act == 3 else 2.0 ** -8) * y.abs()
    (p, q), (ep, eq) = y.chunk(2, 1), e.chunk(2, 1)
    f = torch.nn.functional.gelu(p, approximate="tanh") if act == 2 else \
        torch.nn.functional.silu(p)
    bound = (2.0 ** -8 + 2.0 ** -18) * (f * q).abs() + 1.13 * ep * q.abs() \
        + (f.abs() + ep) * eq
    assert ((got.double() - f * q).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("act", [0, 1, 2, 3])
@pytest.mark.parametrize("tile", range(len(TILES)))
def test_tiles(tile, act):
    """One row and one column tile, ends inside a tile, the shortest K, and so many
    tiles that blocks take three of them, the last turn a part."""
    bm, bn, ahead = TILES[tile]
    if act and bn % 128:
        with pytest.raises(RuntimeError):
            lm_ext().wide_gemm(*operands(64, 64, 1024), tile, act)
        return
    short = 64 * (2 * ahead - 1)
    for M, N, K in [(1, 32, short), (bm - 1, bn - 32, short + 64),
                    (bm + 1, bn + 32, short), (17 * bm + 5, 33 * bn, short)]:
        x, w = operands(M, N, K, K ** -0.5 if act else 1.0)
        check(lm_ext().wide_gemm(x, w, tile, act), x, w, act)
    with pytest.raises(RuntimeError):
        lm_ext().wide_gemm(*operands(64, 64, short - 64), tile, act)


@pytest.mark.gpu
@pytest.mark.parametrize("N", [16, 48, 272])
def test_columns_in_sixteens(N):
    for tile in range(len(TILES)):
        x, w = operands(300, N, 448)
        check(lm_ext().wide_gemm(x, w, tile, 0), x, w, 0)


SPLIT = [(785, 21_248, 1536), (3666, 9888, 768), (8221, 4512, 768)]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SPLIT)
def test_by_the_rules(M, N, K):
    """As models call them: gated or not, and with rows apart."""
    x, w = operands(M, N, K, K ** -0.5)
    assert lm_ext().gemm_ok(x, w) and D.glu_linear_ok(x, w)
    for glu in (False, True):
        tile, rows, rest = lm_ext().gemm_plan(M, N, K, glu)
        assert tile >= 0 and rows < M
    check(D.linear(x, w), x, w, 0)
    check(D.glu_linear(x, w), x, w, 1)


@pytest.mark.gpu
def test_replayed():
    x, w = operands(1024, 10_240, 512)
    assert lm_ext().gemm_plan(1024, 10_240, 512, False)[0] >= 0
    want = D.linear(x, w)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        got = D.linear(x, w)
    for _ in range(3):
        got.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


@pytest.mark.parametrize("glu", [False, True])
def test_plans(glu):
    """Whole tiles apart, tiles that the activation and K allow."""
    apart = 0
    for M in (256, 1000, 2700, 4700, 10_816, 13_800, 44_800):
        for N, K in ((512, 192), (2048, 448), (4096, 4096), (5568, 5888),
                     (28_672, 4096), (32_736, 256)):
            tile, rows, rest = lm_ext().wide_gemm_plan(M, N, K, glu)
            for t in [tile] + [rest] * (rows < M):
                bm, bn, ahead = TILES[t]
                assert K >= 64 * (2 * ahead - 1) and not (glu and bn % 128)
            assert rows == M or (0 < rows < M and rows % TILES[tile][0] == 0)
            apart += rows < M
    assert apart > 3
    assert lm_ext().wide_gemm_plan(1000, 1024, 128, glu)[0] == -1


@pytest.mark.parametrize("M,N,K,glu", [
    (18_556, 1536, 384, False), (2213, 9216, 448, False), (5034, 8192, 512, False),
    (10_626, 2560, 640, False), (14_758, 3072, 384, True), (5595, 4864, 512, True)])
def test_short_products_stay_whole(M, N, K, glu):
    """A launch of its own for the last rows costs more than it saves."""
    assert lm_ext().wide_gemm_plan(M, N, K, glu)[1] == M


@pytest.mark.parametrize("M,N,K", [(8192, 4096, 4096), (8189, 4096, 4096),
                                   (20_480, 8192, 8192), (2048, 16_384, 2048)])
def test_whole_turns_are_the_library_s(M, N, K):
    """Plain products whose tiles of 256 x 256 fill the chip so many times; not those
    of one row more, of short K, or with the activation inside."""
    def ours(m, k=K, glu=False):
        return lm_ext().gemm_sizes(m, N, k, k, glu)

    assert not ours(M) and ours(M, glu=True)
    assert ours(M // 256 * 256 + 257) and ours(M, 1024)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(40, 2048, 1024), (9000, 28_672, 3136)])
def test_rows_gemm_s_own_rules(M, N, K):
    """What is rows_gemm's by its sizes, whatever wide_gemm takes."""
    x, w = (torch.empty(n, K, dtype=BF, device=DEV) for n in (M, N))
    for ok, glu in ((lm_ext().rows_gemm_ok, False), (lm_ext().rows_glu_ok, True)):
        assert ok(x, w) == lm_ext().rows_gemm_sizes(M, N, K, glu) == (M == 40)


@pytest.mark.gpu
@pytest.mark.parametrize("act", [1, 2, 3])
@pytest.mark.parametrize("M,N,K", [
    (257, 6144, 1088), (330, 10_080, 128), (330, 12_288, 192), (300, 16_416, 576),
    (700, 9696, 832), (385, 16_384, 704), (1000, 8864, 576), (1159, 9376, 128),
    (1283, 8128, 1600), (1500, 6176, 1024), (1700, 8192, 256), (2100, 4096, 576)])
def test_rows_gemm_s_gated_tiles(M, N, K, act):
    """Gated products of many rows by rows_gemm.hip, where the rules may take
    wide_gemm.hip."""
    x, w = operands(M, N, K, K ** -0.5)
    check(lm_ext().rows_glu(x, w, act == 2, act != 3), x, w, act)
