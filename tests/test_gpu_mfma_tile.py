"""The matrix-core min-plus tile (mfma_tile.h) at the edges of its digits, chunks and columns.

Bit-exact against the oracle.  Values around 2^22 - 1 are where the digit sums
end and the workgroup turns to integer additions; chunks are 8 deep, columns
are staged four at a time.
"""

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu
INF = O.INF
TOP = (1 << 22) - 2  # largest value that the digits hold


def values(rng, shape, hi, p_inf):
    m = rng.integers(0, hi + 1, shape).astype(np.int32)
    m[rng.random(shape) < 0.1] = hi
    m[rng.random(shape) < p_inf] = INF
    return m


# (where a value the digits do not hold stands: first, middle, last chunk, both operands)
@pytest.mark.parametrize("hi,plant", [(TOP, None), (TOP, "A0"), (TOP, "A"), (TOP, "B-1"),
                                      (TOP + 1, None), (INF - 1, None), (3, None)])
@pytest.mark.parametrize("M,N,K", [(128, 128, 64), (100, 131, 9), (256, 259, 23)])
@pytest.mark.parametrize("accumulate", [False, True])
def test_product_values(gpu_ctx, hi, plant, M, N, K, accumulate):
    rng = np.random.default_rng(M + K + hi)
    A, B = values(rng, (M, K), hi, 0.2), values(rng, (K, N), hi, 0.2)
    C = values(rng, (M, N), INF - 1, 0.3)
    if plant:
        if plant == "B-1":
            B[K - 1, N - 1] = 1 << 22
        else:
            A[M - 1, 0 if plant == "A0" else K // 2] = INF - 1
    dA, dB, dC = gpu_ctx.to_device(A), gpu_ctx.to_device(B), gpu_ctx.to_device(C)
    gpu_ctx.minplus(dA.ptr, K, dB.ptr, N, dC.ptr, N, M, N, K, accumulate)
    gpu_ctx.sync()
    want = O.min_plus_acc(A, B, C) if accumulate else O.min_plus(A, B)
    np.testing.assert_array_equal(dC.get(), want)
    for d in (dA, dB, dC):
        d.free()


@pytest.mark.parametrize("K", [1, 7, 8, 9, 15, 16, 17])
@pytest.mark.parametrize("N", [1, 3, 4, 5, 127, 129])
def test_product_edges(gpu_ctx, K, N):
    M = 97
    rng = np.random.default_rng(100 * K + N)
    A, B = values(rng, (M, K), 5000, 0.3), values(rng, (K, N), 5000, 0.3)
    dA, dB = gpu_ctx.to_device(A), gpu_ctx.to_device(B)
    guard = np.full((M + 1) * N, -5, np.int32)
    dC = gpu_ctx.to_device(guard)
    gpu_ctx.minplus(dA.ptr, K, dB.ptr, N, dC.ptr, N, M, N, K)
    gpu_ctx.sync()
    got = dC.get()
    np.testing.assert_array_equal(got[:M * N].reshape(M, N), O.min_plus(A, B))
    assert (got[M * N:] == -5).all()  # nothing past the last row
    for d in (dA, dB, dC):
        d.free()


@pytest.mark.parametrize("n", [129, 256, 300, 517])
@pytest.mark.parametrize("hi", [1000, 1 << 21, 1 << 26])
def test_closure_values(gpu_ctx, n, hi):
    """The 128-block closure, values below, across and above the digits."""
    rng = np.random.default_rng(n + hi)
    m = values(rng, (n, n), hi, 0.9)
    np.fill_diagonal(m, 0)
    d = gpu_ctx.to_device(m)
    gpu_ctx.set_option("fw_tile", 128)
    try:
        gpu_ctx.fw(d.ptr, n, n)
        gpu_ctx.sync()
    finally:
        gpu_ctx.set_option("fw_tile", 0)
    np.testing.assert_array_equal(d.get(), O.floyd(m))
    d.free()


@pytest.mark.parametrize("sizes", [[449, 512] + [500] * 56, [385, 64, 130, 700] * 16, [321] * 128,
                                   [256] * 511])
@pytest.mark.parametrize("hi,pad", [(1000, 0), (1 << 25, 3)])
def test_batched_pair_passes(gpu_ctx, sizes, hi, pad):
    """Batches with enough tiles for pair passes in 128 x 128 tiles, and two that keep 64 x 64 (jobs
    of 321: half-empty last blocks; 511 jobs of one 128-tile each: too few)."""
    rng = np.random.default_rng(sum(sizes) + hi)
    mats = []
    for n in sizes:
        m = values(rng, (n, n), hi, 0.95)
        np.fill_diagonal(m, 0)
        buf = np.full((n, n + pad), -3, np.int32)
        buf[:, :n] = m
        mats.append((m, gpu_ctx.to_device(buf)))
    gpu_ctx.fw_batched([d.ptr for _, d in mats], sizes, [n + pad for n in sizes])
    for i, (m, d) in enumerate(mats):
        n = m.shape[0]
        got = d.get()
        if i % 8:  # the oracle closes every eighth
            d.free()
            continue
        np.testing.assert_array_equal(got[:, :n], O.floyd(m))
        assert (got[:, n:] == -3).all()
        d.free()


@pytest.mark.parametrize("n", [1, 3, 70, 1023, 1025, 2050])
def test_dense_rows(gpu_ctx, n):
    """Dense matrices from CSRs: row lengths around the 1,024-column pieces, more than 64 arcs in a
    row, duplicates (the last wins), self loops, an unaligned stride."""
    import fastapsp_amd as fa
    rng = np.random.default_rng(n)
    want = np.full((n, n + 1), -8, np.int32)
    want[:, :n] = INF
    ro, col, w = [0], [], []
    for u in range(n):
        k = int(rng.integers(0, 8)) if u % 17 else 150
        c, x = rng.integers(0, n, k), rng.integers(0, 1000, k)
        for a, b in zip(c, x):
            want[u, a] = b
        want[u, u] = 0
        col += list(c)
        w += list(x)
        ro.append(len(col))
    g = fa.DeviceGraph(gpu_ctx, np.array(ro, np.int32), np.array(col, np.int32),
                       np.array(w, np.int32))
    d = gpu_ctx.to_device(np.full((n, n + 1), -8, np.int32))
    gpu_ctx.dense_from_graphs([g], [d.ptr], [n + 1])
    np.testing.assert_array_equal(d.get(), want)
    d.free()
    g.close()
