"""The split-bf16 GEMM tiles (128x128, 64x64) and the clamped edges of the direct ones, where they can
go wrong: rows, columns and K past the tiles, short and ragged K, unaligned rows, split-K, and
operands that the split itself does not settle (infinities, NaN, overflow, values near underflow).

The bound of the ordinary cases: each product of three-part operands is off by at most 2^-25 of its
size, the accumulators add K / 32 roundings of 2^-24, and a 2-norm over normal operands averages them:
3e-7 of the result's norm is above what K <= 1024 can give and below what a dropped bf16 part (2^-18)
would."""
import numpy as np
import pytest

import gpu_util as G
from pulsatrix_amd import native as N

gpu = pytest.mark.gpu

TILES = [N.TILE_128x128_SPLIT, N.TILE_64x64_SPLIT]
DIRECT = [N.TILE_32x64_DIRECT, N.TILE_32x32_DIRECT, N.TILE_32x48_DIRECT]


def product(a, b, ta, tb, tile, splits=1, **more):
    """op(a) op(b) through one forced tile; a and b as stored."""
    m, k = a.shape[::-1] if ta else a.shape
    n = b.shape[0] if tb else b.shape[1]
    da, db, dc = G.dev(a), G.dev(b), G.empty((m, n))
    ws = G.empty((splits * m * n,))
    d = N.GemmDesc()
    d.m, d.n, d.k, d.batch, d.inner, d.kgroups = m, n, k, 1, 1, 1
    d.trans_a, d.trans_b, d.tile, d.splits = int(ta), int(tb), tile, splits
    d.a, d.b, d.c = N.operand(da.data_ptr(), a.shape[1]), N.operand(db.data_ptr(), b.shape[1]), N.operand(dc.data_ptr(), n)
    d.workspace, d.workspace_bytes = ws.data_ptr(), ws.numel() * 4
    for key, v in more.items():
        setattr(d, key, v)
    N.gemm(d, G.stream())
    return G.host(dc)


def stored(x, trans):
    return np.ascontiguousarray(x.T) if trans else x


@gpu
@pytest.mark.parametrize("tile", TILES + DIRECT)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n,k,splits", [(1, 1, 1, 1), (127, 65, 31, 1), (129, 63, 33, 1), (64, 128, 64, 1),
                                          (33, 130, 97, 2), (200, 257, 1000, 3), (65, 64, 160, 1), (3, 2, 1024, 4)])
def test_edges_match_float64(tile, ta, tb, m, n, k, splits):
    rng = np.random.RandomState(m + n + k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    want = a.astype(np.float64) @ b.astype(np.float64)
    got = product(stored(a, ta), stored(b, tb), ta, tb, tile, splits)
    # the direct tiles' fp32 chains round every 4 K steps: up to 1e-6 at K = 1024
    assert np.linalg.norm(got - want) <= (3e-7 if tile in TILES else 1e-6) * np.linalg.norm(want)


@gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("splits", [1, 2])
def test_values_the_split_cannot_hold(tile, splits):
    """Infinities, NaN, products that overflow and operands whose low bf16 parts underflow come out as the
    fp32 tiles give them."""
    rng = np.random.RandomState(7)
    a, b = rng.standard_normal((150, 200)).astype(np.float32), rng.standard_normal((200, 140)).astype(np.float32)
    a[3, 5], a[70, 9], a[100, 1] = np.inf, np.nan, 3.4e38
    b[1, 100], b[17, 66] = 3.0, -np.inf
    a[20] *= np.float32(1e-35)  # a row of results near 1e-34
    with np.errstate(all="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
        want = np.where(np.abs(want) > np.finfo(np.float32).max, np.sign(want) * np.inf, want)
    got = product(a, b, 0, 0, tile, splits)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
    fine = np.isfinite(want)
    scale = np.abs(np.nan_to_num(a)).astype(np.float64) @ np.abs(np.nan_to_num(b)).astype(np.float64)
    assert np.all(np.abs(got - want)[fine] <= 1e-5 * scale[fine])
    assert np.linalg.norm(got[20][fine[20]] - want[20][fine[20]]) <= 1e-6 * np.linalg.norm(want[20][fine[20]])


@gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("where", ["a", "b"])
@pytest.mark.parametrize("small,large", [(3e-31, 1e8), (1e-33, 1e10), (1e-36, 1e20), (1e-38, 1e25), (1e-41, 1e30), (1e-21, 1e-21)])
def test_small_operands(tile, where, small, large):
    """A row of A (a column of B) whose bf16 parts would be subnormal or nothing, against a large other
    operand: no result of the tile is small, and all are as exact as the fp32 tiles give them (subnormal
    ones, of 1e-21 by 1e-21, to their last bits)."""
    rng = np.random.RandomState(11)
    a, b = rng.standard_normal((130, 96)).astype(np.float32), rng.standard_normal((96, 70)).astype(np.float32)
    if where == "a":
        a[129] *= np.float32(small)
        b *= np.float32(large)
    else:
        b[:, 2] *= np.float32(small)
        a *= np.float32(large)
    want = a.astype(np.float64) @ b.astype(np.float64)
    size = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    # 24 fp32 MFMAs of four K steps each round their running sum, which stays below size, by at most 2^-24
    # of it (half of that on average); subnormal products are off by 2^-149 each
    bound = 12 * 2.0 ** -24 * size + 96 * 2.0 ** -149
    for t in (tile, N.TILE_64x64):
        off = np.abs(product(a, b, 0, 0, t) - want) / bound
        print("tile %d: at most %.3g of the bound" % (t, off.max()))
        assert off.max() <= 1.0


@gpu
def test_rows_past_32_bit_offsets():
    """A sliding window over one long row (A^T with a leading dimension of 1): its rows past 2^30 lie past what
    the lanes' 32-bit byte offsets reach from the matrix's start."""
    torch = G.torch_cuda()
    m, k = (1 << 30) + 70, 40
    gen = torch.Generator(device="cuda").manual_seed(2)
    row, b, c = torch.randn(m + k - 1, device="cuda", generator=gen), torch.randn(k, device="cuda", generator=gen), torch.empty(m, device="cuda")
    d = N.GemmDesc()
    d.m, d.n, d.k, d.batch, d.inner, d.kgroups, d.trans_a, d.tile, d.splits = m, 1, k, 1, 1, 1, 1, N.TILE_128x128_SPLIT, 1
    d.a, d.b, d.c = N.operand(row.data_ptr(), 1), N.operand(b.data_ptr(), 1), N.operand(c.data_ptr(), 1)
    N.gemm(d, G.stream())
    for at in (0, (1 << 30) - 128, m - 100):
        x = row[at:at + 100 + k - 1].double()
        want = x.unfold(0, k, 1) @ b.double()
        assert float((c[at:at + 100].double() - want).norm()) <= 3e-7 * float(want.norm())
    del row, c
    torch.cuda.empty_cache()


@gpu
@pytest.mark.parametrize("tile", TILES)
def test_no_less_exact_than_the_fp32_tiles(tile):
    """Against float64 on normal, positive and heavy-tailed operands, beside the fp32 MFMA's direct tile. The
    split tiles stand where one fp32 accumulator ran over the whole of K; the direct tile adds four
    quarters of it, with a quarter of the roundings each and so half the error: the bound is twice its."""
    rng = np.random.RandomState(3)
    for draw in (lambda *s: rng.standard_normal(s), lambda *s: np.abs(rng.standard_normal(s)),
                 lambda *s: rng.standard_normal(s) * np.exp(2.0 * rng.standard_normal(s))):
        a, b = draw(96, 1536).astype(np.float32), draw(1536, 96).astype(np.float32)
        want = a.astype(np.float64) @ b.astype(np.float64)
        err = [np.linalg.norm(product(a, b, 0, 0, t) - want) for t in (tile, N.TILE_32x32_DIRECT)]
        print("split %.3g, fp32 in four K slices %.3g" % tuple(np.array(err) / np.linalg.norm(want)))
        assert err[0] <= 2.0 * err[1]
