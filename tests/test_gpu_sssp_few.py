"""SSSP kernel: LDS queues and their ends (GPU), against Dijkstra.

The kernel keeps the near queue of a workgroup of NT threads in LDS (2 NT
entries, later ones in memory) and the arcs past a vertex's fourth in a second
list (NT / 4 entries).  The graphs reach each side of both, with bands from one
unit to everything at once.
"""
import numpy as np
import pytest

import oracle_lib as O
from fastapsp_amd import INF, synth

pytestmark = pytest.mark.gpu


def graph(kind):
    rng = np.random.default_rng(3)
    if kind == "star":  # one frontier of every vertex: past the LDS queue; a hub of many arcs
        u, v = np.zeros(6000, np.int64), np.arange(1, 6001)
        return 6001, u, v, rng.integers(0, 50, 6000), False
    if kind == "dense":  # 40 arcs a vertex: every entry leaves arcs to the second list
        u = np.repeat(np.arange(3000), 40)
        return 3000, u, rng.integers(0, 3000, u.size), rng.integers(1, 1000, u.size), True
    if kind == "wide":  # unit weights: whole levels in one round
        u = np.repeat(np.arange(20000), 6)
        return 20000, u, rng.integers(0, 20000, u.size), np.ones(u.size, np.int64), True
    if kind == "heavy":  # distances at and past INF
        u = np.arange(400)
        return 401, u, u + 1, np.full(400, INF // 300), True
    if kind == "single":
        return 1, np.zeros(0, np.int64), np.zeros(0, np.int64), np.zeros(0, np.int64), True
    u, v, w = synth.grid_graph(130, 130, 0.05, 0.10, 0, 9, 6)  # five and more arcs, weights of 0
    return 16900, u, v, w, False


@pytest.mark.parametrize("kind", ["star", "dense", "wide", "heavy", "single", "grid"])
@pytest.mark.parametrize("threads,delta,binq", [(1024, 0, 3), (512, 1, 3), (512, 1 << 24, 0),
                                                (256, 0, 3)])
def test_few_sources(gpu_ctx, kind, threads, delta, binq):
    V, u, v, w, directed = graph(kind)
    keep = u != v
    ro, col, wt = synth.to_csr(V, u[keep], v[keep], w[keep], directed)
    src = np.unique(np.array([0, 1, V // 3, V // 2, V - 1], np.int32) % V)
    src = np.concatenate([src, src[:1]]).astype(np.int32)
    if kind == "heavy":
        delta = max(delta, INF // 100)
    dg = gpu_ctx.upload_graph(ro, col, wt)
    ds, out = gpu_ctx.to_device(src), gpu_ctx.alloc((len(src), V))
    try:
        for name, x in (("sssp_threads", threads), ("sssp_delta", delta), ("sssp_bin", binq)):
            gpu_ctx.set_option(name, x)
        dg.sssp(ds.ptr, len(src), out.ptr, V)
    finally:
        for name, x in (("sssp_threads", 0), ("sssp_delta", 0), ("sssp_bin", 3)):
            gpu_ctx.set_option(name, x)
    np.testing.assert_array_equal(out.get(), O.batched_sssp(src, ro, col, wt))
    dg.close()


@pytest.mark.parametrize("count", [1, 256, 257, 512, 513])
def test_source_counts(gpu_ctx, count):
    """Each side of the rule's lines: 1024, 512 and 256 threads."""
    u, v, w = synth.grid_graph(24, 30, 0.05, 0.02, 1, 60, 5)
    ro, col, wt = synth.to_csr(720, u, v, w, False)
    src = (np.arange(count) * 7 % 720).astype(np.int32)
    dg = gpu_ctx.upload_graph(ro, col, wt)
    ds, out = gpu_ctx.to_device(src), gpu_ctx.alloc((count, 720))
    dg.sssp(ds.ptr, count, out.ptr, 720)
    np.testing.assert_array_equal(out.get(), O.batched_sssp(src, ro, col, wt))
    dg.close()
