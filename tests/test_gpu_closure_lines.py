"""Dense closures on both sides of the sizes where the default dispatch changes its launches (256 compute
units): one launch a round up to 16 blocks of 64, phases beyond, blocks of 128 from 35 of them on."""

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu
INF = O.INF


def matrix(n, hi):
    rng = np.random.default_rng(n + hi)
    m = np.full((n, n), INF, np.int32)
    u, v = rng.integers(0, n, 6 * n), rng.integers(0, n, 6 * n)
    m[u, v] = rng.integers(1, hi, u.size)
    np.fill_diagonal(m, 0)
    return m


def closed(gpu_ctx, m, ld, **options):
    n = m.shape[0]
    buf = np.full((n, ld), -9, np.int32)
    buf[:, :n] = m
    d = gpu_ctx.to_device(buf)
    for k, v in options.items():
        gpu_ctx.set_option(k, v)
    try:
        gpu_ctx.fw(d.ptr, n, ld)
        gpu_ctx.sync()
    finally:
        gpu_ctx.set_option("fw_tile", 0)
        gpu_ctx.set_option("fw_lookahead", -1)
    got = d.get()
    d.free()
    assert (got[:, n:] == -9).all()
    return got[:, :n]


@pytest.mark.parametrize("n", [1024, 1025])
@pytest.mark.parametrize("pad", [0, 1])
@pytest.mark.parametrize("hi", [1000, 1 << 24])
def test_round_launches_end(gpu_ctx, n, pad, hi):
    m = matrix(n, hi)
    np.testing.assert_array_equal(closed(gpu_ctx, m, n + pad), O.floyd(m))


@pytest.mark.parametrize("n", [4352, 4353])
@pytest.mark.parametrize("hi", [1000, 1 << 24])
def test_block_sizes_meet(gpu_ctx, n, hi):
    m = matrix(n, hi)
    got = closed(gpu_ctx, m, n)
    for tile in (64, 128):
        np.testing.assert_array_equal(closed(gpu_ctx, m, n, fw_tile=tile), got)
    rows = np.array([0, 1, n // 2, n - 1], np.int32)
    u, v = np.nonzero((m < INF) & ~np.eye(n, dtype=bool))
    ro = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=n))]).astype(np.int32)
    want = O.batched_sssp(rows, ro, v.astype(np.int32), m[u, v])
    np.testing.assert_array_equal(got[rows], want)
