"""SSSP fronts larger than a workgroup's queue in LDS: the queue goes through memory, reordered or not,
and back.  Rows equal to the oracle's."""

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


def random_arcs(V, degree, whi, rng):
    u = np.repeat(np.arange(V), degree)
    v, w = rng.integers(0, V, u.size), rng.integers(1, whi + 1, u.size)
    ro = np.arange(V + 1) * degree
    return ro.astype(np.int32), v.astype(np.int32), w.astype(np.int32)


def star(V, rng):
    """All from the centre (one front of V - 1), and from each leaf to the next."""
    w = np.concatenate([rng.integers(1, 5, V - 1), rng.integers(1, 3, V - 1)])
    col = np.concatenate([np.arange(1, V), np.arange(1, V - 1) + 1, [0]])
    ro = np.concatenate([[0], V - 1 + np.arange(V)])
    return ro.astype(np.int32), col.astype(np.int32), w.astype(np.int32)


# queue room is 512, 1024 or 2048 entries: fronts around, above and far above it; every reordering option
@pytest.mark.parametrize("graph", ["random 1100", "random 6000", "random 30000", "star 514", "star 20000"])
@pytest.mark.parametrize("threads", [256, 512, 1024])
@pytest.mark.parametrize("binq", [0, 1, 2, 3])
def test_wide_fronts(gpu_ctx, graph, threads, binq):
    kind, V = graph.split()
    V = int(V)
    rng = np.random.default_rng(V + threads)
    ro, col, w = star(V, rng) if kind == "star" else random_arcs(V, 7, 40, rng)
    src = np.array([0, V - 1, V // 2], np.int32)
    dg = gpu_ctx.upload_graph(ro, col, w)
    gpu_ctx.set_option("sssp_threads", threads)
    gpu_ctx.set_option("sssp_bin", binq)
    try:
        d_src, out = gpu_ctx.to_device(src), gpu_ctx.alloc((src.size, V))
        dg.sssp(d_src.ptr, src.size, out.ptr, V)
        gpu_ctx.sync()
        got = out.get()
    finally:
        gpu_ctx.set_option("sssp_threads", 0)
        gpu_ctx.set_option("sssp_bin", 3)
    np.testing.assert_array_equal(got, O.batched_sssp(src, ro, col, w))
    d_src.free()
    out.free()
    dg.close()


# beyond two sources a compute unit: 256 threads a source, or 512 from 2^17 vertices on
@pytest.mark.parametrize("side", [362, 363])
def test_threads_by_vertex_count(gpu_ctx, side):
    from fastapsp_amd import synth
    V = side * side
    u, v, w = synth.grid_graph(side, side, 0.10, 0.02, 1, 100, 3)
    ro, col, w = synth.to_csr(V, u, v, w, False)
    src = np.random.default_rng(side).choice(V, 513, replace=False).astype(np.int32)
    dg = gpu_ctx.upload_graph(ro, col, w)
    d_src, out = gpu_ctx.to_device(src), gpu_ctx.alloc((src.size, V))
    dg.sssp(d_src.ptr, src.size, out.ptr, V)
    gpu_ctx.sync()
    got = out.get()
    at = [0, 1, 255, 256, 511, 512]
    np.testing.assert_array_equal(got[at], O.batched_sssp(src[at], ro, col, w))
    d_src.free()
    out.free()
    dg.close()
