"""Values that the digits of the matrix-core tile do not hold, met in the first chunk or a later one: the
tile goes on with integer additions from there.  Bit-exact against the oracle."""

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu
INF = O.INF
BIG = 1 << 23  # above the digits' 2^22 - 2


# chunks are 8 k deep; the first one, its neighbours, the last two (K = 101: they overlap); both operands;
# odd row strides; tiles 5 columns and 70 rows wide at the edges
@pytest.mark.parametrize("k", [0, 7, 8, 15, 16, 50, 92, 93, 100])
@pytest.mark.parametrize("operand,pad", [("A", 0), ("B", 0), ("A", 1), ("B", 3)])
@pytest.mark.parametrize("accumulate", [False, True])
def test_product_turns_at_chunk(gpu_ctx, k, operand, pad, accumulate):
    M, N, K = 198, 261, 101
    rng = np.random.default_rng(1000 * k + pad)
    A = rng.integers(0, 5000, (M, K + pad)).astype(np.int32)
    B = rng.integers(0, 5000, (K, N + pad)).astype(np.int32)
    A[rng.random(A.shape) < 0.2] = INF
    B[rng.random(B.shape) < 0.2] = INF
    if operand == "A":
        A[rng.integers(0, M, 3), k] = BIG
        A[M - 1, k] = INF - 1
    else:
        B[k, rng.integers(0, N, 3)] = BIG
        B[k, N - 1] = INF - 1
    C = rng.integers(0, 9000, (M, N + pad)).astype(np.int32)
    C[rng.random(C.shape) < 0.3] = INF
    dA, dB, dC = gpu_ctx.to_device(A), gpu_ctx.to_device(B), gpu_ctx.to_device(C)
    gpu_ctx.minplus(dA.ptr, K + pad, dB.ptr, N + pad, dC.ptr, N + pad, M, N, K, accumulate)
    gpu_ctx.sync()
    got = dC.get()
    a, b, c = (np.ascontiguousarray(x) for x in (A[:, :K], B[:, :N], C[:, :N]))
    np.testing.assert_array_equal(got[:, :N], O.min_plus_acc(a, b, c) if accumulate else O.min_plus(a, b))
    np.testing.assert_array_equal(got[:, N:], C[:, N:])
    for d in (dA, dB, dC):
        d.free()


def closure_input(n, hi, late, rng):
    """Sparse weights up to hi; late: small ones, and large ones only on the arcs of every 64-block's
    last vertex, which a block's products meet in their last chunk."""
    m = rng.integers(1, 1000 if late else hi + 1, (n, n)).astype(np.int32)
    if late:
        m[63::64, :] = rng.integers(BIG, 2 * BIG, m[63::64, :].shape)
        m[:, 63::64] = rng.integers(BIG, 2 * BIG, m[:, 63::64].shape)
    m[rng.random((n, n)) > max(0.02, 8 / n)] = INF
    np.fill_diagonal(m, 0)
    return m


# The 64-block closure in phases: panels whose result is also an operand, phase 3 with the next diagonal
# inside, rows and columns past the last block.  Look-ahead keeps small n on this path.
@pytest.mark.parametrize("n,pad,lookahead", [(70, 0, 1), (128, 0, 1), (131, 1, 1), (200, 0, 1), (257, 2, 1),
                                             (1025, 0, 0), (1025, 1, 0), (1088, 0, 0), (1283, 1, 0)])
@pytest.mark.parametrize("hi,late", [(1 << 21, False), (1 << 26, False), (0, True)])
def test_closure_in_64_blocks(gpu_ctx, n, pad, lookahead, hi, late):
    rng = np.random.default_rng(n + pad + hi)
    m = closure_input(n, hi, late, rng)
    buf = np.full((n, n + pad), -9, np.int32)
    buf[:, :n] = m
    d = gpu_ctx.to_device(buf)
    gpu_ctx.set_option("fw_tile", 64)
    gpu_ctx.set_option("fw_lookahead", lookahead)
    try:
        gpu_ctx.fw(d.ptr, n, n + pad)
        gpu_ctx.sync()
    finally:
        gpu_ctx.set_option("fw_tile", 0)
        gpu_ctx.set_option("fw_lookahead", -1)
    got = d.get()
    np.testing.assert_array_equal(got[:, :n], O.floyd(m))
    assert (got[:, n:] == -9).all()
    d.free()


# Boundary block updates (fewer than 32 parts: no coarse level): every block past the digits, or some of
# its border positions only; lists below and above 16 positions, several chunks
@pytest.mark.parametrize("side,K", [(24, 5), (48, 6)])
@pytest.mark.parametrize("share", [1.0, 0.03])
@pytest.mark.parametrize("tile", [0, 64, 128])
def test_boundary_blocks(gpu_ctx, side, K, share, tile):
    from fastapsp_amd import synth
    V = side * side
    u, v, w = synth.grid_graph(side, side, 0.05, 0.02, 1, 100, side + K)
    rng = np.random.default_rng(side)
    w = np.where(rng.random(len(w)) < share, rng.integers(1 << 20, 1 << 23, len(w)), w).astype(np.int32)
    ro, col, w = synth.to_csr(V, u, v, w, False)
    gid = (np.arange(V) * K // V + 1).astype(np.int32)
    pc = O.precondition(K, gid, ro, col)
    dg = gpu_ctx.upload_graph(ro, col, w)
    dg.set_partition(gid, pc["st2ed"], pc["ed2st"])
    assert dg.build_index()
    gpu_ctx.set_option("bidx_tile", tile)
    try:
        for ids in ([2], list(range(1, K + 1))):
            outs = [gpu_ctx.alloc((int(pc["ver_num"][p]), V)) for p in ids]
            dg.subgraph_solve_batch([int(pc["ver_off"][p]) for p in ids],
                                    [int(pc["ver_num"][p]) for p in ids],
                                    [int(pc["bdy_num"][p]) for p in ids], [o.ptr for o in outs], V)
            for p, o in zip(ids, outs):
                if p <= 2:
                    np.testing.assert_array_equal(o.get(), O.run_part(p, ro, col, w, gid, pc))
                o.free()
    finally:
        gpu_ctx.set_option("bidx_tile", 0)
    dg.close()
