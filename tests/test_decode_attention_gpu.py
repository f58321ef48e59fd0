"""pxk_decode_attention against float64 at the edges of its forms: head_dims that one, several or no
128-bit vectors of a thread hold, the first and last keys of a chunk, windows that cut a chunk, and
caches on both sides of the 64 chunks that the merge weighs at once. Keys past the position hold NaN."""
import numpy as np
import pytest

import gpu_util as G
from pulsatrix_amd import native as N


def run(n, H, Hkv, D, cap, pos, window, masked=()):
    """masked: keys of every sequence whose scores are all -inf."""
    rng = np.random.RandomState(D + pos)
    q = rng.standard_normal((n, H, D)).astype(np.float32)
    k, v = (rng.standard_normal((n, cap, Hkv, D)).astype(np.float32) for _ in range(2))
    k[:, pos + 1:], v[:, pos + 1:] = np.nan, np.nan
    if len(masked):
        q[..., 0] = np.abs(q[..., 0]) + 1.0
        k[:, list(masked), :, 0] = -np.inf
    lo = max(0, pos + 1 - window) if window else 0
    torch = G.torch_cuda()
    dq, dk, dv, ctx = G.dev(q), G.dev(k), G.dev(v), G.empty((n, H, D))
    dpos = G.keep(torch.tensor([pos], dtype=torch.int32, device="cuda"))
    need = N.pxk().pxk_decode_attention_workspace(n, H, D, cap)
    ws = G.empty((need // 4,))
    N.call("pxk_decode_attention", G.ptr(dq), G.ptr(dk), G.ptr(dv), cap * Hkv * D, G.ptr(ctx), G.ptr(dpos), n, H, Hkv, D,
           window, cap, D ** -0.5, G.ptr(ws), need, G.stream())
    grp = H // Hkv
    kk = np.repeat(k[:, lo:pos + 1].astype(np.float64), grp, axis=2)
    vv = np.repeat(v[:, lo:pos + 1].astype(np.float64), grp, axis=2)
    s = np.einsum("nhd,njhd->nhj", q.astype(np.float64), kk) * D ** -0.5
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    want, size = np.einsum("nhj,njhd->nhd", p, vv), np.einsum("nhj,njhd->nhd", p, np.abs(vv))
    # a score is off by D roundings of terms that add up to a few units, a weight by that and an ulp or two
    assert np.all(np.abs(G.host(ctx).reshape(n, H, D) - want) <= 1e-5 * size)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [4, 6, 40, 60, 64, 68, 80, 100, 128, 132, 192, 252, 256, 260])
@pytest.mark.parametrize("pos", [0, 1, 62, 63, 64, 129])
def test_head_dims_and_positions(D, pos):
    run(2, 4, 2, D, 131, pos, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [40, 64, 256])
@pytest.mark.parametrize("pos,window", [(5, 1), (70, 7), (100, 64), (130, 65), (130, 200)])
def test_windows(D, pos, window):
    run(3, 2, 1, D, 140, pos, window)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [6, 40, 64, 256, 320])
@pytest.mark.parametrize("cap,pos,masked", [(131, 130, range(64)), (131, 130, range(3, 64)), (300, 299, range(64, 192)), (300, 299, range(192, 299)),
                                            (70, 69, range(64, 70)), (4160, 4159, range(128, 256))])
def test_chunks_of_scores_minus_infinity(cap, pos, masked, D):
    """A chunk whose every score is -inf counts for nothing, like one that holds no key."""
    run(2, 2, 1, D, cap, pos, 0, masked)


@pytest.mark.gpu
@pytest.mark.parametrize("cap,pos", [(4096, 4095), (4097, 4096), (4160, 300), (257, 256), (300, 10)])
@pytest.mark.parametrize("D", [64, 320])
def test_long_caches(cap, pos, D):
    run(1, 2, 1, D, cap, pos, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [132, 256])
@pytest.mark.parametrize("n,cap", [(1, 4096), (1, 4097), (4, 1088)])
def test_wide_heads_in_small_and_large_grids(n, cap, D):
    """Head_dims past 128 on both sides of the 512 workgroups up to which a chunk is held in registers."""
    run(n, 8, 2, D, cap, cap - 1, 0)
