"""The boundary index's matrix-core tiles at their edges: border lists longer than one LDS piece, lists
shorter than a chunk, values past the digits.  Rows equal to the oracle's per-part pipeline."""

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


def solve_all(gpu_ctx, ro, col, w, gid, K):
    """Row blocks of every part through one batched call, and the oracle's preconditioning."""
    V = len(ro) - 1
    pc = O.precondition(K, gid, ro, col)
    dg = gpu_ctx.upload_graph(ro, col, w)
    dg.set_partition(gid, pc["st2ed"], pc["ed2st"])
    assert dg.build_index()
    ids = list(range(1, K + 1))
    outs = [gpu_ctx.alloc((int(pc["ver_num"][p]), V)) for p in ids]
    dg.subgraph_solve_batch([int(pc["ver_off"][p]) for p in ids], [int(pc["ver_num"][p]) for p in ids],
                            [int(pc["bdy_num"][p]) for p in ids], [o.ptr for o in outs], V)
    got = [o.get() for o in outs]
    for o in outs:
        o.free()
    dg.close()
    return got, pc


def random_digraph(V, degree, whi, seed):
    rng = np.random.default_rng(seed)
    u = np.repeat(np.arange(V), degree)
    v = rng.integers(0, V, V * degree)
    keep = u != v
    key = np.unique(u[keep] * V + v[keep])
    u, v = key // V, key % V
    w = rng.integers(1, whi + 1, u.size).astype(np.int32)
    ro = np.zeros(V + 1, np.int32)
    np.cumsum(np.bincount(u, minlength=V), out=ro[1:])
    return ro, v.astype(np.int32), w


# 900 vertices a part, nearly all on its border: lists of ~900 positions (two pieces); 521 and 520
# around the longest list that stays in one piece; 1 << 24: integer additions
@pytest.mark.parametrize("V,K,whi", [(1800, 2, 100), (1800, 2, 1 << 24), (1042, 2, 50), (1040, 2, 50),
                                     (1500, 3, 255)])
def test_long_border_lists(gpu_ctx, V, K, whi):
    ro, col, w = random_digraph(V, 6, whi, V + K)
    gid = (np.arange(V) * K // V + 1).astype(np.int32)
    got, pc = solve_all(gpu_ctx, ro, col, w, gid, K)
    for p in range(1, K + 1):
        np.testing.assert_array_equal(got[p - 1], O.run_part(p, ro, col, w, gid, pc))


# a path of cliques: borders of one vertex, lists of one or two positions
def test_short_border_lists(gpu_ctx):
    K, n = 9, 30
    V = K * n
    arcs = []
    rng = np.random.default_rng(4)
    for p in range(K):
        for i in range(n):
            for j in rng.integers(0, n, 4):
                if i != j:
                    arcs.append((p * n + i, p * n + int(j)))
        if p:
            arcs += [(p * n, p * n - 1), (p * n - 1, p * n)]
    arcs = sorted(set(arcs))
    u = np.array([a for a, _ in arcs])
    ro = np.zeros(V + 1, np.int32)
    np.cumsum(np.bincount(u, minlength=V), out=ro[1:])
    col = np.array([b for _, b in arcs], np.int32)
    w = rng.integers(1, 1000, len(arcs)).astype(np.int32)
    gid = (np.arange(V) // n + 1).astype(np.int32)
    got, pc = solve_all(gpu_ctx, ro, col, w, gid, K)
    for p in range(1, K + 1):
        np.testing.assert_array_equal(got[p - 1], O.run_part(p, ro, col, w, gid, pc))


# Graphs with the index's coarse level (32 parts and more), through whole calls and one part a call; two
# components; directed arcs one way only between regions; a graph without locality keeps the index alone.
def region_graph(kind):
    from fastapsp_amd import synth
    if kind == "grid":
        u, v, w = synth.grid_graph(72, 72, 0.10, 0.02, 1, 100, 8)
        return (*synth.to_csr(72 * 72, u, v, w, False), 64)
    if kind == "large weights":
        u, v, w = synth.grid_graph(60, 60, 0.10, 0.02, 1, 1 << 23, 9)
        return (*synth.to_csr(3600, u, v, w, False), 40)
    if kind == "components":
        u, v, w = synth.grid_graph(64, 64, 0.05, 0.0, 1, 9, 10)
        keep = (u // 64 < 30) == (v // 64 < 30)  # the rows below 30 and the others
        return (*synth.to_csr(4096, u[keep], v[keep], w[keep], False), 48)
    if kind == "one way":
        u, v, w = synth.grid_graph(60, 60, 0.05, 0.02, 1, 50, 11)
        a, b, x = np.concatenate([u, v]), np.concatenate([v, u]), np.concatenate([w, w])
        keep = (a // 60 < b // 60) | (a // 60 == b // 60) | (a % 7 == 0)  # upwards in every 7th column
        return (*synth.to_csr(3600, a[keep], b[keep], x[keep], True), 36)
    return (*random_digraph(2000, 3, 50, 12), 40)  # no locality


@pytest.mark.parametrize("kind", ["grid", "large weights", "components", "one way", "no locality"])
def test_coarse_level(gpu_ctx, kind):
    import fastapsp_amd as fa
    ro, col, w, K = region_graph(kind)
    V = len(ro) - 1
    with fa.Graph.from_csr(ro, col, w.astype(np.float32), K) as g:
        g.preCondition()
        gid = g.getGraphId()
    got, pc = solve_all(gpu_ctx, ro, col, w, gid, K)
    for p in range(1, K + 1, 5):
        np.testing.assert_array_equal(got[p - 1], O.run_part(p, ro, col, w, gid, pc))
    # one part a call, from a graph whose index is new: the 32nd call makes the coarse level
    dg = gpu_ctx.upload_graph(ro, col, w)
    dg.set_partition(gid, pc["st2ed"], pc["ed2st"])
    sizes = []
    for p in range(1, K + 1):
        n, b = int(pc["ver_num"][p]), int(pc["bdy_num"][p])
        out = gpu_ctx.alloc((n, V))
        dg.subgraph_solve_batch([int(pc["ver_off"][p])], [n], [b], [out.ptr], V)
        np.testing.assert_array_equal(out.get(), got[p - 1])
        out.free()
        sizes.append(dg.index_info()[1])
    assert (sizes[30] < sizes[31]) == (kind != "no locality")
    dg.set_partition(gid, pc["st2ed"], pc["ed2st"])  # drops both
    assert dg.index_info() == (0, 0)
    dg.close()


# Parts that share launches: without boundary, nothing but boundary, one vertex, more rows than a tile;
# the products with fewer than 8 k, and with none.
def test_uneven_parts_share_launches(gpu_ctx):
    rng = np.random.default_rng(21)
    sizes = [40, 12, 12, 1, 300, 150]
    first = np.concatenate([[0], np.cumsum(sizes)])
    arcs = []
    for q, n in enumerate(sizes):
        for i in range(1, n):
            if q not in (1, 2):  # each vertex hangs on an earlier one of its part
                arcs.append((first[q] + rng.integers(0, i), first[q] + i))
    arcs += [(first[1] + i, first[2] + j) for i in range(12) for j in range(12) if (i + j) % 3 == 0]
    arcs += [(first[4] + 7, first[5] + 3), (first[4] + 200, first[5] + 90), (first[2] + 4, first[4])]
    u, v = np.array(arcs).T
    V = int(first[-1])
    from fastapsp_amd import synth
    ro, col, w = synth.to_csr(V, u, v, rng.integers(1, 90, u.size), False)
    gid = np.repeat(np.arange(len(sizes)), sizes).astype(np.int32) + 1
    got, pc = solve_all(gpu_ctx, ro, col, w, gid, len(sizes))
    for p in range(1, len(sizes) + 1):
        np.testing.assert_array_equal(got[p - 1], O.run_part(p, ro, col, w, gid, pc))
