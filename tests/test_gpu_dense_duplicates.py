"""Rows of a dense matrix whose arcs repeat columns: the last arc in CSR order holds, within 64 arcs and
across them, in every 1,024-column piece; a self loop never does."""

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 65, 1025, 2049])
@pytest.mark.parametrize("order", ["up", "down"])
def test_last_duplicate_holds(gpu_ctx, n, order):
    import fastapsp_amd as fa
    rng = np.random.default_rng(n)
    targets = np.array(sorted({0, 1, n // 2, n - 1}))
    ro, col, w = [0], [], []
    want = np.full((n, n), O.INF, np.int32)
    for u in range(n):
        k = (0, 1, 2, 63, 64, 65, 130)[u % 7]
        c = targets[rng.integers(0, targets.size, k)]
        x = np.arange(1, k + 1) if order == "up" else np.arange(k, 0, -1)
        for a, b in zip(c, x):
            want[u, a] = b
        want[u, u] = 0
        col += list(c)
        w += list(x)
        ro.append(len(col))
    g = fa.DeviceGraph(gpu_ctx, np.array(ro, np.int32), np.array(col, np.int32), np.array(w, np.int32))
    d = gpu_ctx.to_device(np.full((n, n), -8, np.int32))
    gpu_ctx.dense_from_graphs([g], [d.ptr], [n])
    np.testing.assert_array_equal(d.get(), want)
    d.free()
    g.close()
