"""The split-bf16 GEMM tiles (128x128, 64x64) and the clamped edges of the direct ones, where they can
go wrong: rows, columns and K past the tiles, short and ragged K, unaligned rows, split-K, causal ranges,
K-groups and batch strides, leading dimensions past 32-bit offsets, and operands that the split itself
does not settle (infinities, NaN, overflow) or settles by its scale (values near underflow).

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
    """Infinities, NaN and products that overflow come out as the fp32 tiles give them, and small results to
    their last bits."""
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
@pytest.mark.parametrize("causal", [N.CAUSAL_NONE, N.CAUSAL_TRI, N.CAUSAL_K_LE_M, N.CAUSAL_K_GE_M])
@pytest.mark.parametrize("kgroups,k", [(1, 256), (1, 201), (3, 64), (3, 75)])
@pytest.mark.parametrize("splits", [1, 2])
def test_causal_ranges_groups_and_strides(tile, causal, kgroups, k, splits):
    """Batches of 2 x 2 with B shared by the inner two (a KV head), K-groups strided apart, and the causal
    ranges, whose tiles neither read K outside their range (NaN here) nor compute above the diagonal."""
    m, n = (k, 70) if causal in (N.CAUSAL_K_LE_M, N.CAUSAL_K_GE_M) else (201, 140)
    rng = np.random.RandomState(k + causal)
    a, b = rng.standard_normal((4, kgroups, m, k)).astype(np.float32), rng.standard_normal((2, kgroups, k, n)).astype(np.float32)
    rows, cols, bm = np.arange(m)[:, None], np.arange(k)[None], 128 if tile == N.TILE_128x128_SPLIT else 64
    if causal == N.CAUSAL_K_LE_M:
        a[..., cols > rows] = 0.0
        a[..., cols >= (rows // bm + 1) * bm] = np.nan
    if causal == N.CAUSAL_K_GE_M:
        a[..., cols < rows] = 0.0
        a[..., cols < rows // bm * bm] = np.nan
    want = np.einsum("bgmk,bgkn->bmn", np.nan_to_num(a).astype(np.float64), np.repeat(b, 2, axis=0).astype(np.float64))
    da, db, dc = G.dev(a), G.dev(b), G.empty((4, m, n))
    ws = G.empty((splits * 4 * m * n,))
    d = N.GemmDesc()
    d.m, d.n, d.k, d.batch, d.inner, d.kgroups, d.causal, d.tile, d.splits = m, n, k, 4, 2, kgroups, causal, tile, splits
    d.a = N.operand(da.data_ptr(), k, 2 * kgroups * m * k, kgroups * m * k, 1, m * k)
    d.b = N.operand(db.data_ptr(), n, kgroups * k * n, kgroups * k * n, 2, k * n)
    d.c = N.operand(dc.data_ptr(), n, 2 * m * n, m * n, 1)
    d.workspace, d.workspace_bytes = ws.data_ptr(), ws.numel() * 4
    N.gemm(d, G.stream())
    got = G.host(dc).reshape(4, m, n)
    keep = np.tril(np.ones((m, n), bool)) if causal == N.CAUSAL_TRI else np.ones((m, n), bool)
    assert np.linalg.norm((got - want)[:, keep]) <= 3e-7 * np.linalg.norm(want[:, keep])


@gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_leading_dimensions_past_32_bit_offsets(tile, ta, tb):
    """Rows 2^22 elements apart and further are loaded element by element."""
    torch = G.torch_cuda()
    m, n, k, ld = 70, 65, 40, (1 << 22) + 3
    gen = torch.Generator(device="cuda").manual_seed(3)
    A, B = (torch.zeros(r, ld, device="cuda") for r in ((k if ta else m), (n if tb else k)))
    a, b = A[:, :m if ta else k], B[:, :k if tb else n]
    a.copy_(torch.randn(a.shape, device="cuda", generator=gen))
    b.copy_(torch.randn(b.shape, device="cuda", generator=gen))
    c = torch.empty(m, n, device="cuda")
    d = N.GemmDesc()
    d.m, d.n, d.k, d.batch, d.inner, d.kgroups, d.trans_a, d.trans_b, d.tile, d.splits = m, n, k, 1, 1, 1, ta, tb, tile, 1
    d.a, d.b, d.c = N.operand(A.data_ptr(), ld), N.operand(B.data_ptr(), ld), N.operand(c.data_ptr(), n)
    N.gemm(d, G.stream())
    a, b = a.cpu().double().numpy(), b.cpu().double().numpy()
    want = (a.T if ta else a) @ (b.T if tb else b)
    assert np.linalg.norm(c.cpu().double().numpy() - want) <= 3e-7 * np.linalg.norm(want)
    del A, B
    torch.cuda.empty_cache()


@gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("k", [96, 101])
def test_values_the_split_cannot_hold_after_the_prologue(tile, bias, k):
    """The divided operand with an infinity and a NaN, and quotients and products that overflow the split's
    range: the tiles computed again divide too. Rows and columns without them stay exact."""
    m, n, eps = 140, 70, 1e-6
    rng = np.random.RandomState(k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((n, k)).astype(np.float32)
    z = (rng.uniform(0.5, 1.5, (m, k)) * rng.choice([-1.0, 1.0], (m, k))).astype(np.float32)
    zb = rng.uniform(-0.2, 0.2, k).astype(np.float32) if bias else np.zeros(k, np.float32)
    x = rng.standard_normal((m, n)).astype(np.float32)
    a[3, 5], a[70, 9], a[100, 1], a[139, k - 1] = np.inf, np.nan, 1e30, 1e32
    zz = z.astype(np.float64) + zb
    q = a / (zz + eps * np.where(zz >= 0, 1.0, -1.0))
    with np.errstate(all="ignore"):
        want = x * (q @ b.T.astype(np.float64))
        scale = np.abs(x) * (np.abs(q) @ np.abs(b.T).astype(np.float64))
    dc, keep = G.empty((m, n)), [G.dev(v) for v in (a, b, z, x, zb)]
    d = N.GemmDesc()
    d.m, d.n, d.k, d.batch, d.inner, d.kgroups, d.trans_b, d.tile, d.splits = m, n, k, 1, 1, 1, 1, tile, 1
    d.prologue, d.epilogue, d.eps = N.PRO_DIV_STAB, N.EPI_MUL_X, eps
    d.a, d.b, d.z, d.x = (N.operand(t.data_ptr(), w) for t, w in zip(keep, (k, k, k, n)))
    if bias:
        d.z_bias = N.operand(keep[4].data_ptr(), 0)
    d.c = N.operand(dc.data_ptr(), n)
    N.gemm(d, G.stream())
    got = G.host(dc).reshape(m, n)
    fine = np.isfinite(want)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
    # a quotient takes a reciprocal within an ulp and two roundings, the products up to K / 4 more
    assert np.all(np.abs(got - want)[fine] <= (4 + k / 4) * 2.0 ** -24 * scale[fine])


@gpu
@pytest.mark.parametrize("tile,fp32", [(N.TILE_128x128_SPLIT, N.TILE_128x128), (N.TILE_64x64_SPLIT, N.TILE_64x64)])
@pytest.mark.parametrize("k", [64, 576, 1536, 8192])
def test_no_less_exact_than_the_fp32_tiles(tile, fp32, k):
    """Against float64 on normal, positive and heavy-tailed operands, beside the fp32 tile of the same size,
    whose place each split tile takes."""
    rng = np.random.RandomState(3)
    for draw in (lambda *s: rng.standard_normal(s), lambda *s: np.abs(rng.standard_normal(s)),
                 lambda *s: rng.standard_normal(s) * np.exp(2.0 * rng.standard_normal(s))):
        a, b = draw(96, k).astype(np.float32), draw(k, 96).astype(np.float32)
        want = a.astype(np.float64) @ b.astype(np.float64)
        err = [np.linalg.norm(product(a, b, 0, 0, t) - want) for t in (tile, fp32)]
        print("split %.3g, fp32 %.3g" % tuple(np.array(err) / np.linalg.norm(want)))
        assert err[0] <= err[1]
