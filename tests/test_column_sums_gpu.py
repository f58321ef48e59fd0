"""pxk_column_sums at the edges of its 16-column workgroups and 64-row steps, and of the widths that go to
one thread a column, against float64: sums of up to 1024 terms a lane in fp32 stay within 1e-6 of the
column's absolute sum."""
import numpy as np
import pytest

import gpu_util as G
from pulsatrix_amd import native as N


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols", [(0, 5), (1, 1), (16, 300), (17, 300), (63, 16), (64, 17), (65, 15), (511, 33), (513, 100), (4096, 2048),
                                       (16384, 31), (17, 17407), (17, 17408), (18, 17408), (30, (1 << 19) - 1), (513, 1 << 19), (700, (1 << 19) - 1)])
@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_column_sums(rows, cols, beta):
    rng = np.random.RandomState(rows + cols)
    x, old = rng.standard_normal((rows, cols)).astype(np.float32), rng.standard_normal(cols).astype(np.float32)
    out = G.dev(old)
    N.call("pxk_column_sums", G.ptr(G.dev(x)) if rows else None, G.ptr(out), rows, cols, beta, G.stream())
    want = beta * old.astype(np.float64) + x.astype(np.float64).sum(0)
    bound = 1e-6 * (np.abs(x.astype(np.float64)).sum(0) + np.abs(old))
    assert np.all(np.abs(G.host(out) - want) <= bound)
