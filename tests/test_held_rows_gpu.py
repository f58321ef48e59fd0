"""The row kernels that hold a row in registers, at the edges of their shapes (a wave or a workgroup a
row, float4 or single floats, rows past 8192 columns) against float64. A row's terms are summed in
fp32 over at most 512 terms a lane before a tree over lanes, exponentials are good to an ulp or two and
each result takes a handful of roundings: 1e-6 of the sum of the terms' magnitudes bounds them."""
import ctypes

import numpy as np
import pytest

import gpu_util as G
from pulsatrix_amd import native as N

COLS = [1, 3, 63, 64, 65, 127, 128, 129, 132, 255, 256, 257, 260, 508, 511, 512, 513, 516, 1023, 1024, 1025, 1028, 1535, 1536, 1537, 2047,
        2048, 2049, 2052, 3071, 3073, 4095, 4096, 4097, 4100, 6143, 6145, 8191, 8192, 8193, 8196]


def _call(name, *args):
    args = [ctypes.c_int64(v) if isinstance(v, int) else v for v in args]
    N.check(getattr(N.pxk(), name)(*args, G.stream()))


def _dev(a, offset):
    """`a` on the GPU, `offset` floats past a 16-byte boundary."""
    flat = G.dev(np.concatenate([np.zeros(offset, np.float32), np.asarray(a, np.float32).ravel()]))
    return flat[offset:]


@pytest.mark.gpu
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("cols", COLS)
def test_held_rows(cols, offset):
    rows = 7
    rng = np.random.RandomState(cols)
    x, g, w = (rng.standard_normal(s).astype(np.float32) for s in ((rows, cols), (rows, cols), (cols,)))
    rms = np.sqrt((x.astype(np.float64) ** 2).mean(1) + 1e-5).astype(np.float32)
    X, Gr, W, R = (a.astype(np.float64) for a in (x, g, w, rms))
    E = np.exp(X - X.max(1, keepdims=True))
    P = E / E.sum(1, keepdims=True)
    dx, dg, dw, dr = _dev(x, offset), _dev(g, offset), _dev(w, offset), G.dev(rms)
    guard = 5  # a row past the end stays as it was
    outs = [G.dev(np.full(offset + rows * cols + guard, 7.0, np.float32)) for _ in range(4)]
    p, dp, gx, gt = (o[offset:] for o in outs)
    lse = G.dev(np.full(rows + guard, 7.0, np.float32))
    _call("pxk_softmax_rows", G.ptr(dx), G.ptr(p), rows, cols)
    _call("pxk_logsumexp_rows", G.ptr(dx), G.ptr(lse), rows, cols)
    _call("pxk_softmax_rows_backward", G.ptr(dx), G.ptr(dg), G.ptr(dp), rows, cols)
    _call("pxk_rms_norm_backward", G.ptr(dg), G.ptr(dw), G.ptr(dx), G.ptr(dr), G.ptr(gx), G.ptr(gt), rows, cols)
    norm, got_rms = G.dev(np.full(offset + rows * cols + guard, 7.0, np.float32)), G.dev(np.full(rows + guard, 7.0, np.float32))
    _call("pxk_rms_norm_forward", G.ptr(dx), G.ptr(dw), G.ptr(norm[offset:]), G.ptr(got_rms), rows, cols, ctypes.c_float(1e-5))
    outs += [norm, got_rms]
    for o in outs + [lse]:
        assert np.all(G.host(o)[-guard:] == 7.0)
    host = lambda o: G.host(o)[:rows * cols].reshape(rows, cols).astype(np.float64)  # noqa: E731
    assert np.all(np.abs(host(p) - P) <= 2e-6 * P)
    want = X.max(1) + np.log(E.sum(1))
    assert np.all(np.abs(G.host(lse)[:rows] - want) <= 1e-6 * (1.0 + np.abs(want)))
    want = np.sqrt((X ** 2).mean(1) + 1e-5)
    assert np.all(np.abs(G.host(got_rms)[:rows] - want) <= 1e-6 * want)
    assert np.all(np.abs(host(norm[offset:]) - W * X / want[:, None]) <= 1e-6 * np.abs(W * X / want[:, None]))
    dot, size = (X * Gr).sum(1, keepdims=True), np.abs(X * Gr).sum(1, keepdims=True)
    assert np.all(np.abs(host(dp) - X * (Gr - dot)) <= 1e-6 * np.abs(X) * (np.abs(Gr) + size))
    Rc = R[:, None]
    assert np.all(np.abs(host(gt) - Gr * X / Rc) <= 1e-6 * np.abs(Gr * X / Rc))
    dot, size = (Gr * W * X).sum(1, keepdims=True), np.abs(Gr * W * X).sum(1, keepdims=True)
    scale = X / (cols * Rc ** 3)
    assert np.all(np.abs(host(gx) - (Gr * W / Rc - scale * dot)) <= 1e-6 * (np.abs(Gr * W / Rc) + np.abs(scale) * size))


@pytest.mark.gpu
@pytest.mark.parametrize("cols", [5, 260, 1100, 2052, 8192])
def test_held_softmax_extremes(cols):
    """Masks of -inf and of the type's lowest value, whole masked rows, +inf and NaN: as IEEE gives
    them in exp(x - max) / sum."""
    x = np.random.RandomState(cols).standard_normal((6, cols)).astype(np.float32)
    x[0, cols // 2:] = -np.inf
    x[1, cols // 2:] = np.finfo(np.float32).min
    x[2, :] = np.finfo(np.float32).min
    x[3, :] = -np.inf
    x[4, -1] = np.inf
    x[5, 0] = np.nan
    with np.errstate(invalid="ignore"):
        X = x.astype(np.float64)
        E = np.exp(X - np.fmax.reduce(X, axis=1, keepdims=True))
        P = E / E.sum(1, keepdims=True)
        L = np.fmax.reduce(X, axis=1) + np.log(E.sum(1))
    d, p, lse = _dev(x, 0), G.empty((6, cols)), G.empty((6,))
    _call("pxk_softmax_rows", G.ptr(d), G.ptr(p), 6, cols)
    _call("pxk_logsumexp_rows", G.ptr(d), G.ptr(lse), 6, cols)
    np.testing.assert_allclose(G.host(p), P, rtol=2e-6, atol=0)
    np.testing.assert_allclose(G.host(lse), L, rtol=1e-6, atol=1e-6)
    _call("pxk_softmax_rows", G.ptr(d), G.ptr(d), 6, cols)  # in place
    assert np.array_equal(G.host(d).reshape(6, cols), G.host(p), equal_nan=True)


@pytest.mark.gpu
def test_more_rows_than_workgroups():
    """2^24 rows of more than 1024 columns: one workgroup a row would be a launch of 2^32 threads."""
    torch = G.torch_cuda()
    rows, cols = 1 << 24, 1028
    x, lse = torch.zeros(rows, cols, device="cuda"), torch.empty(rows, device="cuda")
    some = torch.tensor([0, 1, rows // 2, rows - 2, rows - 1], device="cuda")
    x[some] = torch.randn(len(some), cols, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    want = x[some].double()
    _call("pxk_logsumexp_rows", G.ptr(x), G.ptr(lse), rows, cols)
    _call("pxk_softmax_rows", G.ptr(x), G.ptr(x), rows, cols)
    assert float((lse[some] - want.logsumexp(1)).abs().max()) <= 1e-5
    assert float((x[some] / want.softmax(1) - 1).abs().max()) <= 2e-6
    assert float((lse[2:1000] - float(np.log(cols))).abs().max()) <= 1e-5
    del x
    torch.cuda.empty_cache()
