"""pxk_attention_softmax and pxk_attention_lrp_scores at the spans where the held rows begin
and end (2048 and 4096 keys) and below, with windows and without a causal mask, against
float64: exponentials and sums of up to 64 terms a lane in fp32, 1e-5 of the terms' size."""
import numpy as np
import pytest

import gpu_util as G
from pulsatrix_amd import native as N


@pytest.mark.gpu
@pytest.mark.parametrize("l,causal,window", [(256, 1, 0), (257, 1, 0), (320, 1, 0), (600, 0, 0), (700, 1, 300), (1024, 1, 0),
                                             (1025, 1, 0), (2048, 1, 0), (2049, 0, 0), (2500, 1, 1100), (2500, 1, 2200), (4096, 1, 0),
                                             (4097, 1, 0), (4200, 1, 4095), (300, 1, 40)])
def test_attention_rows(l, causal, window):
    scale, eps = 0.125, 1e-6
    rng = np.random.RandomState(l + window)
    raw, ra = (rng.standard_normal((1, l, l)).astype(np.float32) * 4 for _ in range(2))
    i, j = np.arange(l)[:, None], np.arange(l)[None]
    vis = (j <= i if causal else np.ones((l, l), bool)) & ((j + window > i) if window and causal else True)
    raw[0][~vis] = ra[0][~vis] = np.nan  # masked entries are not read
    x = np.where(vis, scale * raw[0].astype(np.float64), -np.inf)
    P = np.exp(x - x.max(1, keepdims=True))
    P /= P.sum(1, keepdims=True)
    dr, da, dp, ds = G.dev(raw), G.dev(ra), G.empty((l, l)), G.empty((l, l))
    N.call("pxk_attention_softmax", G.ptr(dr), G.ptr(dp), 1, l, scale, causal, window, G.stream())
    got = G.host(dp)
    assert np.all(got[~vis] == 0.0) and np.all(np.abs(got - P) <= 1e-5 * P)
    N.call("pxk_attention_lrp_scores", G.ptr(da), G.ptr(dp), G.ptr(dr), G.ptr(ds), 1, l, scale, eps, causal, window, G.stream())
    r, o, p = np.where(vis, ra[0], 0).astype(np.float64), np.where(vis, raw[0], 1).astype(np.float64), got.astype(np.float64)
    den = 2 * o + eps * np.where(o >= 0, 1.0, -1.0)
    want = np.where(vis, scale * o * (r - p * r.sum(1, keepdims=True)) / den, 0.0)
    size = np.abs(scale * o) * (np.abs(r) + p * np.abs(r).sum(1, keepdims=True)) / np.abs(den)
    s = G.host(ds)
    assert np.all(s[~vis] == 0.0) and np.all(np.abs(s - want) <= 1e-5 * size + 1e-30)
    N.call("pxk_attention_lrp_scores", G.ptr(da), G.ptr(dp), G.ptr(dr), G.ptr(da), 1, l, scale, eps, causal, window, G.stream())
    assert np.array_equal(G.host(da)[0], s)  # in place
