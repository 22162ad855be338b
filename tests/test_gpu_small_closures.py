"""Closures around the sizes where the dense closure changes its launches: one block, one launch per
round (up to 1.5 tiles per compute unit), three launches per round; odd strides and a positive
diagonal, which a pivot must not relax through.  Bit-exact against the oracle."""

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu
INF = O.INF


@pytest.mark.parametrize("n", [1, 2, 5, 63, 64, 65, 66, 127, 129, 191, 449, 1216, 1217])
@pytest.mark.parametrize("pad,diag", [(0, 0), (1, 3)])
def test_closure_sizes(gpu_ctx, n, pad, diag):
    if n > 1000 and pad:
        pytest.skip("one layout is enough at the large sizes")
    rng = np.random.default_rng(n)
    m = rng.integers(1, 1000, (n, n)).astype(np.int32)
    m[rng.random((n, n)) < (0.5 if n < 100 else 0.97)] = INF
    np.fill_diagonal(m, diag)
    buf = np.full((n, n + pad), -9, np.int32)
    buf[:, :n] = m
    d = gpu_ctx.to_device(buf)
    gpu_ctx.fw(d.ptr, n, n + pad)
    gpu_ctx.sync()
    got = d.get()
    np.testing.assert_array_equal(got[:, :n], O.floyd(m))
    assert (got[:, n:] == -9).all()
    d.free()
